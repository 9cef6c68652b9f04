"""GPU: gradients of tile lists that several workgroups composite.

- the undo adjoint starts at log(1 - alpha) of the rendered image on a split list
  as on a whole one: against the float64 oracle started from the renderer's own
  image, within four times the distance of the float32 oracle from it.  Pixels
  down to T = 3e-6, where the rounding of alpha moves the gradients by 1.5e-4 to
  5e-4 of those from an exact image;
- an L1 step has the image of one pass over each list, and the adjoint of it;
- both adjoints with a near offset, in calls of many tiles, under the scene-major
  order and through the autotuner; a view alone and in a batch;
- segment buffers sized by what calls with short segments can need.
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


def _scene(scale=1.0):
    rng = np.random.default_rng(7)
    s = make_scene(uniform_points(4000, rng), rng)
    s["densities"] = (s["densities"] * scale).astype(np.float32)
    return s


def _renderer(s, w=W, h=H, **kw):
    from rmeshvk_amd import RMeshRenderer

    return RMeshRenderer(s["vertices"], s["indices"], s["base_colors"], s["densities"], s["color_grads"],
                         s["circumdata"], w, h, device_id=0, **kw)


def _longest(ref):
    r = np.asarray(ref["ranges"]).reshape(-1, 2).astype(np.int64)
    return int((r[:, 1] - r[:, 0]).max())


# the second camera is a wide angle: a large view with the mesh in a few of its tiles
@pytest.mark.parametrize("ts,w,h,fov,scale", [(8, W, H, 50.0, 1.8), (12, W, H, 50.0, 1.8), (16, W, H, 50.0, 1.8),
                                              (32, W, H, 50.0, 1.8), (12, 280, 280, 140.0, 1.6)])
def test_undo_starts_at_the_image_alpha(ts, w, h, fov, scale):
    s, cam = _scene(scale), fibonacci_cameras(2, 3.0, fov, w, h)[1]
    ref = orc.render(s, cam, w, h, ts)
    assert _longest(ref) > 2 * (6 * ts * ts)
    assert 1e-6 < (1.0 - ref["rgba"][..., 3].astype(np.float64)).min() < 1e-5
    dl = np.random.default_rng(ts).normal(0, 1e-2, (h, w, 4)).astype(np.float32)
    r = _renderer(s, w, h, tile_size=ts)
    img = np.asarray(r.forward_tiled(*cam)).reshape(h, w, 4)
    g = r.backward(dl)
    f64 = {k: (np.asarray(v, np.float64) if np.asarray(v).dtype == np.float32 else v) for k, v in s.items()}
    go = orc.backward(f64, cam, w, h, ref["sorted_vals"], ref["ranges"], img.astype(np.float64), dl.astype(np.float64),
                      ts, dtype=np.float64)
    g32 = orc.backward(s, cam, w, h, ref["sorted_vals"], ref["ranges"], img, dl, ts)
    for k in KEYS:
        assert _rel(g[k], go[k]) <= 4 * _rel(g32[k], go[k]), (k, _rel(g[k], go[k]), _rel(g32[k], go[k]))


@pytest.mark.parametrize("mode", ["undo", "checkpoint"])
@pytest.mark.parametrize("kind", ["plain", "saturating"])
@pytest.mark.parametrize("ts", [8, 12, 16, 32])
def test_l1_step_composites_in_list_order(ts, kind, mode):
    """The L1 gradient is the sign of image - target, so its image has the
    rounding of one pass over each list.  Towards the image of such a pass (the
    aux forward's) nothing is left: loss and gradients 0; and towards a far
    target the gradients are the unsplit lists'."""
    s, cam = _scene(), fibonacci_cameras(2, 3.0, 50.0, W, H)[1]
    if kind == "saturating":
        x = s["vertices"].reshape(-1, 3)[s["indices"].reshape(-1, 4).astype(int)].mean(1)[:, 0]
        s["densities"] = (s["densities"] * np.where(x > 0.1, 30.0, np.where(x < -0.3, 0.5, 6.0))).astype(np.float32)
    ref = orc.render(s, cam, W, H, ts)
    assert _longest(ref) > 2 * (6 * ts * ts)
    assert ((1.0 - ref["rgba"][..., 3]).min() < 1e-6) == (kind == "saturating") and ref["rgba"].max() < 20.0
    r = _renderer(s, tile_size=ts)
    r.set_adjoint_mode(mode)
    img = np.asarray(r.forward_tiled(*cam, render_aux=True)[0]).reshape(H, W, 4)
    assert r.train_step(*cam, np.ascontiguousarray(img[..., :3]), 0.0, 0.0, 0.0, 0) == 0.0
    np.testing.assert_array_equal(r.read_buffer(0, H * W * 4).reshape(H, W, 4), img)
    for k, v in r.gradients().items():
        assert not np.any(v), k
    gt = np.random.default_rng(3).uniform(20.0, 30.0, (H, W, 3)).astype(np.float32)  # brighter than any pixel
    for _ in range(2):
        r.train_step(*cam, gt, 0.0, 0.0, 0.0, 0)
        g = r.gradients()
    dl = np.concatenate([np.full((H, W, 3), -1.0 / (W * H)), np.zeros((H, W, 1))], -1).astype(np.float32)
    if mode == "checkpoint":
        fw = orc.forward(s, cam, W, H, ref["sorted_vals"], ref["ranges"], ts, want_checkpoints=True)
        go = orc.backward(s, cam, W, H, ref["sorted_vals"], ref["ranges"], fw["rgba"], dl, ts, checkpoints=fw)
    else:
        f64 = {k: (np.asarray(v, np.float64) if np.asarray(v).dtype == np.float32 else v) for k, v in s.items()}
        go = orc.backward(f64, cam, W, H, ref["sorted_vals"], ref["ranges"], img.astype(np.float64),
                          dl.astype(np.float64), ts, dtype=np.float64)
    for k in ("d_vertices", "d_densities", "d_color_grads"):
        assert _rel(g[k], go[k]) <= 1e-3, (k, _rel(g[k], go[k]))


@pytest.mark.parametrize("mode", ["undo", "checkpoint"])
@pytest.mark.parametrize("min_t", [0.5, 3.0])
@pytest.mark.parametrize("ts", [8, 12, 16, 32])
def test_near_offset(ts, min_t, mode):
    """min_t shifts the forward's ray parameter only; the adjoint of a split list
    starts its segments from that forward's states.  The bounds of the unsplit
    path: image 1e-4, gradients 1e-3 relative L2."""
    s, cam = _scene(), fibonacci_cameras(2, 3.0, 50.0, W, H)[1]
    ref = orc.render(s, cam, W, H, ts, min_t=min_t)
    assert _longest(ref) > 2 * (6 * ts * ts)
    dl = np.random.default_rng(ts).normal(0, 1e-2, (H, W, 4)).astype(np.float32)
    r = _renderer(s, tile_size=ts)
    r.set_adjoint_mode(mode)
    r.set_min_t(min_t)
    img = np.asarray(r.forward_tiled(*cam)).reshape(H, W, 4)
    assert np.abs(img - ref["rgba"]).max() <= 1e-4
    g = r.backward(dl)
    if mode == "checkpoint":
        fw = orc.forward(s, cam, W, H, ref["sorted_vals"], ref["ranges"], ts, min_t=min_t, want_checkpoints=True)
        go = orc.backward(s, cam, W, H, ref["sorted_vals"], ref["ranges"], fw["rgba"], dl, ts, checkpoints=fw)
    else:
        f64 = {k: (np.asarray(v, np.float64) if np.asarray(v).dtype == np.float32 else v) for k, v in s.items()}
        go = orc.backward(f64, cam, W, H, ref["sorted_vals"], ref["ranges"], img.astype(np.float64),
                          dl.astype(np.float64), ts, dtype=np.float64)
    for k in KEYS:
        assert _rel(g[k], go[k]) <= 1e-3, (k, _rel(g[k], go[k]))


@pytest.mark.parametrize("mode", ["undo", "checkpoint"])
@pytest.mark.parametrize("ts,w,fov", [(8, 328, 140.0), (12, 480, 145.0), (16, 640, 145.0)])
def test_calls_of_many_tiles(ts, w, fov, mode):
    """Above 1,536 work items, where the segments hold six pairs per pixel: the mesh
    in a few of the tiles of a wide angle.  Image 2e-4 (two float32 evaluations, each
    up to 5.3e-5 from float64 here), gradients 1e-3 relative L2, or four times the
    float32 oracle's own error where that is more (vertices far from the axis)."""
    s, cam = _scene(), fibonacci_cameras(2, 3.0, fov, w, w)[1]
    ref = orc.render(s, cam, w, w, ts)
    assert len(ref["ranges"].reshape(-1, 2)) > 1536 and _longest(ref) > 2 * (6 * ts * ts)
    dl = np.random.default_rng(ts).normal(0, 1e-2, (w, w, 4)).astype(np.float32)
    r = _renderer(s, w, w, tile_size=ts)
    r.set_adjoint_mode(mode)
    img = np.asarray(r.forward_tiled(*cam)).reshape(w, w, 4)
    assert np.abs(img - ref["rgba"]).max() <= 2e-4
    g = r.backward(dl)
    f64 = {k: (np.asarray(v, np.float64) if np.asarray(v).dtype == np.float32 else v) for k, v in s.items()}
    go = orc.backward(f64, cam, w, w, ref["sorted_vals"], ref["ranges"], img.astype(np.float64), dl.astype(np.float64),
                      ts, dtype=np.float64)
    g32 = orc.backward(s, cam, w, w, ref["sorted_vals"], ref["ranges"], img, dl, ts)
    for k in KEYS:
        assert _rel(g[k], go[k]) <= max(1e-3, 4 * _rel(g32[k], go[k])), (k, _rel(g[k], go[k]))


def test_a_thumbnail_scene_does_not_size_the_segments():
    """Segment buffers are sized by the pairs that a call with short segments can
    have, not by all of a renderer that has a small view."""
    from rmeshvk_amd import MultiSceneRenderer, RMeshRenderer

    rng = np.random.default_rng(5)
    big, small = make_scene(uniform_points(40000, rng), rng), make_scene(uniform_points(300, rng), rng)
    cams = fibonacci_cameras(4, 3.0, 50.0, 512, 512)
    one = RMeshRenderer(big["vertices"], big["indices"], big["base_colors"], big["densities"], big["color_grads"],
                        big["circumdata"], 512, 512, device_id=0, max_views=4)
    one.forward_batched(cams, copy_out=False)
    assert one.pair_count() > 2_000_000
    thumb = _renderer(small, 64, 64)
    thumb.forward_tiled(*fibonacci_cameras(1, 3.0, 50.0, 64, 64)[0])
    both = MultiSceneRenderer([dict(big, width=512, height=512, max_views=4), dict(small, width=64, height=64, max_views=1)])
    both.forward([4, 1], cams + fibonacci_cameras(1, 3.0, 50.0, 64, 64))
    # (what the two hold apart, the larger pair buffer's growth step and the rest of a few MB)
    assert both.device_bytes() <= 1.1 * (one.device_bytes() + thumb.device_bytes())


def test_segments_in_scene_major_order():
    from rmeshvk_amd import MultiSceneRenderer

    a, b = _scene(0.2), _scene(1.0)
    cams = fibonacci_cameras(3, 3.0, 50.0, W, H)
    got = []
    for order in ("interleaved", "by_scene"):
        r = MultiSceneRenderer([dict(s, width=W, height=H, max_views=2) for s in (a, b)])
        r.set_scene_order(order)
        r.set_targets([2, 1], [np.full((n, H, W, 3), 0.4, np.float32) for n in (2, 1)])
        r.train_step([2, 1], cams, 1, 0.0, 0.0, 0.0, 0.0)
        got.append((r.read_buffer(0, 3 * H * W * 4), r.gradients()))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    for k, v in got[0][1].items():
        assert _rel(got[1][1][k], v) <= 1e-5, k


def test_segments_through_the_autotuner():
    s, cam = _scene(0.2), fibonacci_cameras(2, 3.0, 50.0, W, H)[1]
    gt = np.full((1, H, W, 3), 0.4, np.float32)
    r = _renderer(s)
    r.set_targets(gt)
    r.autotune([cam], reps=1)
    r.train_step_batched([cam], 1, 0.0, 0.0, 0.0)
    fresh = _renderer(s, tile_size=r.get_tuning()[0])
    fresh.set_tuning(*r.get_tuning())
    fresh.train_step(*cam, gt[0], 0.0, 0.0, 0.0, 1)
    for k, v in fresh.gradients().items():
        assert _rel(r.gradients()[k], v) <= 1e-5, k


def test_the_autotuner_times_a_geometry_once():
    """Forward 6 at tile 16 and adjoint 10 are variant 0's geometries: accepted, and
    never what the autotuner keeps (with both timed it kept either by chance)."""
    s, cam = _scene(0.2), fibonacci_cameras(2, 3.0, 50.0, W, H)[1]
    r = _renderer(s, tile_size=16)
    r.set_targets(np.full((1, H, W, 3), 0.4, np.float32))
    imgs = []
    for f, b in ((0, 0), (6, 10)):
        r.set_tuning(16, f, b)
        imgs.append(r.forward_tiled(*cam))
    np.testing.assert_array_equal(*imgs)
    for _ in range(4):
        ts, f, b = r.autotune([cam], reps=1)["tuning"]
        assert b != 10 and (ts, f) != (16, 6)


@pytest.mark.parametrize("mode", ["undo", "checkpoint"])
def test_a_view_alone_and_in_a_batch(mode):
    """Alone (484 tiles) a view's lists are split at one pair per pixel, among eight
    (3,872) at six: the same image to the rounding of the joined sums (1e-6 a
    channel of order 1, bound 1e-5), and the gradients to what that moves them."""
    s = _scene()
    cams = fibonacci_cameras(8, 3.0, 50.0, 256, 256)
    gts = np.random.default_rng(5).random((8, 256, 256, 3)).astype(np.float32)
    rb, r1 = _renderer(s, 256, 256, max_views=8), _renderer(s, 256, 256)
    for r in (rb, r1):
        r.set_adjoint_mode(mode)
    rb.set_targets(gts)
    rb.train_step_batched(cams, 1, 0.0, 0.0, 0.0)
    images = rb.read_buffer(0, 8 * 256 * 256 * 4).reshape(8, 256, 256, 4)
    total = {}
    for i, (c, gt) in enumerate(zip(cams, gts)):
        r1.train_step(*c, gt, 0.0, 0.0, 0.0, 1)
        assert np.abs(r1.read_buffer(0, 256 * 256 * 4).reshape(256, 256, 4) - images[i]).max() <= 1e-5
        for k, v in r1.gradients().items():
            total[k] = total.get(k, 0.0) + np.asarray(v, np.float64)
    for k, v in rb.gradients().items():
        assert _rel(v, total[k]) <= 2e-5, (k, _rel(v, total[k]))
