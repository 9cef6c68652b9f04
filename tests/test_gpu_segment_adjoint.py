"""GPU: gradients of tile lists that several workgroups composite.

- the undo adjoint starts at log(1 - alpha) of the rendered image on a split list
  as on a whole one: against the float64 oracle started from the renderer's own
  image, within four times the distance of the float32 oracle from it.  Pixels
  down to T = 3e-6, where the rounding of alpha moves the gradients by 1.5e-4 to
  5e-4 of those from an exact image.
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
