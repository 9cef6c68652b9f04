"""GPU: tile lists longer than a segment (6 pairs per pixel of the tile, one in
views of at most 512 tiles), which several workgroups composite, against the
oracle's single pass over each list.

- images within 1e-4 max-abs and checkpointed gradients within 1e-3 relative L2
  of the float32 oracle, the bounds of the unsegmented path, at every tile size,
  with lists of a few and of many segments, in a light scene, in one where no
  pixel saturates but some come close, and in one where pixels saturate in the
  first segment, in later ones and never (the segments from there on are
  composited again);
- the undo mode's gradients within the same bound of the float64 oracle;
- a batch, replayed as a graph, gives every view's image bit for bit and the sum
  of the views' gradients.
"""

import numpy as np
import pytest

from oracle import oracle as orc
from rmeshvk_amd.camera import fibonacci_cameras
from rmeshvk_amd.scenes import make_scene, uniform_points

pytestmark = pytest.mark.gpu

W, H = 40, 28  # partial tiles on both sides at every tile size
KEYS = ("d_vertices", "d_densities", "d_color_grads", "d_base_colors")


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _scene(kind):
    rng = np.random.default_rng(7)
    s = make_scene(uniform_points(4000, rng), rng)
    x = s["vertices"].reshape(-1, 3)[s["indices"].reshape(-1, 4).astype(int)].mean(1)[:, 0]
    scale = {"light": 0.2, "plain": 1.0, "saturating": np.where(x > 0.1, 30.0, np.where(x < -0.3, 0.5, 6.0))}[kind]
    s["densities"] = (s["densities"] * scale).astype(np.float32)
    return s


def _renderer(s, w=W, h=H, **kw):
    from rmeshvk_amd import RMeshRenderer

    return RMeshRenderer(s["vertices"], s["indices"], s["base_colors"], s["densities"], s["color_grads"],
                         s["circumdata"], w, h, device_id=0, **kw)


def _longest(ref):
    r = np.asarray(ref["ranges"]).reshape(-1, 2).astype(np.int64)
    return int((r[:, 1] - r[:, 0]).max())


@pytest.mark.parametrize("kind", ["light", "plain", "saturating"])
@pytest.mark.parametrize("ts", [8, 12, 16, 32])
def test_segmented_lists_match_oracle(kind, ts):
    s, cam = _scene(kind), fibonacci_cameras(2, 3.0, 50.0, W, H)[1]
    ref = orc.render(s, cam, W, H, ts)
    assert _longest(ref) > 2 * (6 * ts * ts)
    t_end = 1.0 - ref["rgba"][..., 3]
    assert (t_end.min() < 1e-6) == (kind == "saturating")
    dl = np.random.default_rng(ts).normal(0, 1e-2, (H, W, 4)).astype(np.float32)
    fw = orc.forward(s, cam, W, H, ref["sorted_vals"], ref["ranges"], ts, want_checkpoints=True)
    go = orc.backward(s, cam, W, H, ref["sorted_vals"], ref["ranges"], fw["rgba"], dl, ts, checkpoints=fw)
    r = _renderer(s, tile_size=ts)
    r.set_adjoint_mode("checkpoint")
    for _ in range(2):  # the second pass starts from what the first left
        img = r.forward_tiled(*cam)
        assert np.abs(img - ref["rgba"]).max() <= 1e-4
        g = r.backward(dl)
        for k in KEYS:
            assert _rel(g[k], go[k]) <= 1e-3, (k, _rel(g[k], go[k]))
    r.set_adjoint_mode("undo")
    img = r.forward_tiled(*cam)
    assert np.abs(img - ref["rgba"]).max() <= 1e-4
    g = r.backward(dl)
    # The undo starts from log(1 - alpha): 1 - alpha carries 6e-8 of the rounding of
    # alpha, a share of T that the oracle takes from the exact image, and for a
    # saturated pixel from the renderer's own alpha.
    f64 = {k: (np.asarray(v, np.float64) if np.asarray(v).dtype == np.float32 else v) for k, v in s.items()}
    fw = orc.forward(f64, cam, W, H, ref["sorted_vals"], ref["ranges"], ts, dtype=np.float64)
    sat = 1.0 - fw["rgba"][..., 3] < np.exp(-13.8)
    start = np.where(sat[..., None], np.asarray(img, np.float64).reshape(H, W, 4), fw["rgba"])
    go = orc.backward(f64, cam, W, H, ref["sorted_vals"], ref["ranges"], start, dl.astype(np.float64), ts,
                      dtype=np.float64)
    for k in KEYS:
        assert _rel(g[k], go[k]) <= 1e-3, (k, _rel(g[k], go[k]))


@pytest.mark.parametrize("kind", ["plain", "saturating"])
@pytest.mark.parametrize("ts,w", [(8, 200), (12, 280), (16, 376)])
def test_segmented_lists_of_a_large_view_match_oracle(kind, ts, w):
    """Views of more than 512 tiles, the mesh in a few of them (a wide angle: seen
    from far away the float32 slabs lose digits on either side).  Image bound: the
    float32 oracle is up to 8.6e-5 from its float64 evaluation here, so two float32
    evaluations may be 2e-4 apart."""
    s, cam = _scene(kind), fibonacci_cameras(2, 3.0, 140.0, w, w)[1]
    ref = orc.render(s, cam, w, w, ts)
    assert len(ref["ranges"].reshape(-1, 2)) > 512 and _longest(ref) > 2 * (6 * ts * ts)
    dl = np.random.default_rng(ts).normal(0, 1e-2, (w, w, 4)).astype(np.float32)
    fw = orc.forward(s, cam, w, w, ref["sorted_vals"], ref["ranges"], ts, want_checkpoints=True)
    go = orc.backward(s, cam, w, w, ref["sorted_vals"], ref["ranges"], fw["rgba"], dl, ts, checkpoints=fw)
    r = _renderer(s, w, w, tile_size=ts)
    r.set_adjoint_mode("checkpoint")
    img = r.forward_tiled(*cam)
    assert np.abs(img - ref["rgba"]).max() <= 2e-4
    g = r.backward(dl)
    for k in KEYS:
        assert _rel(g[k], go[k]) <= 1e-3, (k, _rel(g[k], go[k]))


@pytest.mark.parametrize("mode", ["undo", "checkpoint"])
def test_segmented_batch_and_graph_replays(mode):
    s = _scene("saturating")
    cams = fibonacci_cameras(3, 3.0, 50.0, W, H)
    gts = np.random.default_rng(2).random((3, H, W, 3)).astype(np.float32)
    rb = _renderer(s, max_views=3)
    rb.set_adjoint_mode(mode)
    rb.set_targets(gts)
    rb.set_graph_mode(True)
    r1 = _renderer(s)
    r1.set_adjoint_mode(mode)
    images = np.stack([np.asarray(r1.forward_tiled(*c)).reshape(H, W, 4) for c in cams])
    total = {}
    for c, gt in zip(cams, gts):
        r1.train_step(*c, gt, 0.0, 0.0, 0.0, 1)
        for k, v in r1.gradients().items():
            total[k] = total.get(k, 0.0) + np.asarray(v, np.float64)
    for _ in range(4):
        rb.train_step_batched(cams, 1, 0.0, 0.0, 0.0, 0.0)
        np.testing.assert_array_equal(rb.read_buffer(0, 3 * H * W * 4).reshape(3, H, W, 4), images)
        for k, v in rb.gradients().items():
            assert _rel(v, total[k]) <= 1e-5, (k, _rel(v, total[k]))
