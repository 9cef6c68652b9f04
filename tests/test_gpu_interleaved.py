"""GPU: calls of different kinds on one renderer, in a scene whose tile lists are
split over several workgroups (more than one pair per pixel of the tile).

- backward and forward_error after a graph replay that an aux or interval forward
  came before (those order whole tiles, the replay (tile, segment) items) equal a
  fresh renderer's within 1e-4, where a tile taken twice or left out is of the
  order of 1;
- the interval adjoint is refused after a tiled call, whose lists are not its own.
"""

import numpy as np
import pytest

from rmeshvk_amd.camera import fibonacci_cameras
from rmeshvk_amd.scenes import make_scene, uniform_points

pytestmark = pytest.mark.gpu

W, H = 60, 44
TOL = 1e-4


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.fixture(scope="module")
def scene():
    rng = np.random.default_rng(11)
    s = make_scene(uniform_points(4000, rng), rng)
    s["densities"] = (s["densities"] * 0.2).astype(np.float32)  # no pixel near saturation
    return s


def _renderer(s, **kw):
    from rmeshvk_amd import RMeshRenderer

    return RMeshRenderer(s["vertices"], s["indices"], s["base_colors"], s["densities"], s["color_grads"],
                         s["circumdata"], W, H, device_id=0, **kw)


def _targets(n=1):
    return np.random.default_rng(1).random((n, H, W, 3)).astype(np.float32)


def _dl():
    return np.random.default_rng(2).normal(0, 1e-2, (H, W, 4)).astype(np.float32)


def _same(got, want):
    for k, v in want.items():
        if np.any(v):
            assert _rel(got[k], v) <= TOL, (k, _rel(got[k], v))
        else:
            assert not np.any(got[k]), k


CAMS = fibonacci_cameras(2, 3.0, 50.0, W, H)


@pytest.mark.parametrize("mode", ["undo", "checkpoint"])
@pytest.mark.parametrize("loss", [0, 1])
@pytest.mark.parametrize("between", ["aux", "interval", "two views"])
@pytest.mark.parametrize("ts", [8, 12, 16])
def test_adjoint_and_error_after_a_replay(scene, ts, between, loss, mode):
    cam = CAMS[1]
    pe, se = (np.ascontiguousarray(x) for x in np.random.default_rng(4).random((2, H, W)).astype(np.float32))
    r = _renderer(scene, tile_size=ts, max_views=2)
    r.set_adjoint_mode(mode)
    r.set_targets(_targets(2))
    r.set_graph_mode(True)
    for _ in range(3):  # eager, captured, replayed
        r.train_step_batched([cam], loss, 0.0, 0.0, 0.0)
    if between == "aux":
        r.forward_tiled(*CAMS[0], render_aux=True)
    elif between == "interval":
        r.forward_interval_tiled(*CAMS[0])
    else:
        r.forward_batched(CAMS)
    r.train_step_batched([cam], loss, 0.0, 0.0, 0.0)
    fresh = _renderer(scene, tile_size=ts)
    fresh.set_adjoint_mode(mode)
    fresh.forward_tiled(*cam)
    _same(r.backward(_dl()), fresh.backward(_dl()))
    (err, count), (want, want_count) = r.forward_error(pe, se), fresh.forward_error(pe, se)
    assert _rel(err, want) <= TOL
    np.testing.assert_array_equal(count[:, 0], want_count[:, 0])


@pytest.mark.parametrize("between", ["forward_tiled", "forward_batched", "train_step", "train_step_batched"])
def test_interval_adjoint_after_a_tiled_call_is_refused(scene, between):
    r = _renderer(scene)
    r.set_targets(_targets())
    r.forward_interval_tiled(*CAMS[1])
    {"forward_tiled": lambda: r.forward_tiled(*CAMS[1]),
     "forward_batched": lambda: r.forward_batched(CAMS[1:]),
     "train_step": lambda: r.train_step(*CAMS[1], _targets()[0], 0.0, 0.0, 0.0, 1),
     "train_step_batched": lambda: r.train_step_batched(CAMS[1:], 1, 0.0, 0.0, 0.0)}[between]()
    with pytest.raises(ValueError, match="preceding forward_interval_tiled"):
        r.backward_interval_tiled(_dl())
