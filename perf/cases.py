"""The measured cases: what programs that use this renderer have it do.

A case is one call (or the pair of calls that a program makes together) of the
public API on a seeded scene.  Scenes are Delaunay meshes of uniform or
clustered points as in the repository's configurations; the seed turns the
mesh (a rotation keeps it Delaunay) and draws every parameter and target
image.  Kinds:

  render    forward_tiled, one view, image to the host (a viewer's call)
  views     forward_batched, images left in the device buffer
  train     train_step, the per-view call of the reference's API, host target
  batch     train_step_batched over all views, graph-replayed
  multi     MultiSceneRenderer.train_step over scenes of uneven size
  autograd  RMeshModule forward + backward on GPU tensors
  interval  forward_interval_tiled + backward_interval_tiled
  densify   forward_tiled with aux outputs + forward_error

Training kinds return the loss, the gradients and the updated weights (the
renderer's own device buffers).
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from rmeshvk_amd import MultiSceneRenderer, RMeshRenderer, _lib
from rmeshvk_amd.autograd import RMeshModule
from rmeshvk_amd.camera import fibonacci_cameras
from rmeshvk_amd.scenes import circumspheres, cluster_points, delaunay_tets, uniform_points

# learning rates late in a run: the benchmark's (vertices, densities, colour
# gradients, SH) after a decay of 1/100 (SH 1/25)
LR = (1e-6, 1e-4, 1e-5, 1e-4)


def _case(name, kind, points, clusters, sh, views, width, height, tile, **more):
    return {"name": name, "kind": kind, "points": points, "clusters": clusters, "sh": sh, "views": views,
            "width": width, "height": height, "tile": tile, "loss": more.get("loss", 0),
            "adjoint": more.get("adjoint", "undo"), "fwd": more.get("fwd", 0), "bwd": more.get("bwd", 0)}


def listed():
    return [
        # the smallest call: a viewer redrawing a small mesh (the repository's smallest configuration)
        _case("view_small", "render", 2000, 0, -1, 1, 256, 256, 12),
        # evaluation of several views of an ordinary scene
        _case("views_8", "views", 10000, 0, 3, 8, 512, 512, 12),
        # rendering a large clustered scene in full HD
        _case("views_hd", "views", 100000, 8, 3, 2, 1920, 1080, 16),
        # the reference's own training loop on a small mesh: one view a step, launch bound
        _case("train_small", "train", 2000, 0, -1, 1, 256, 256, 12, loss=1),
        # the same loop on a large scene with SH colours, at the default tuning
        _case("train_view", "train", 60000, 8, 3, 1, 800, 800, 12),
        # batched training of an ordinary scene (8 views at 512 x 512)
        _case("batch_8", "batch", 10000, 0, 3, 8, 512, 512, 12),
        # the repository's benchmark step (squared loss), with the tuning its autotuner keeps there
        _case("batch_16", "batch", 200000, 8, 3, 16, 800, 800, 16, loss=1, fwd=6, bwd=10),
        # training towards saturated pixels: the checkpointed adjoint, low SH degree, squared loss
        _case("batch_checkpoint", "batch", 50000, 4, 1, 4, 640, 480, 16, loss=1, adjoint="checkpoint"),
        # many scenes of uneven size, resolution and SH degree in one step
        _case("multi", "multi", 40000, 6, 3, 2, 512, 512, 16),
        # a torch training program's forward and backward on GPU tensors
        _case("autograd", "autograd", 20000, 0, -1, 1, 512, 512, 12, loss=1),
        # the interval renderer's forward and adjoint, an odd image size
        _case("interval", "interval", 50000, 8, -1, 1, 637, 479, 12),
        # the densification pass: aux outputs and per-tet error statistics, an odd image size
        _case("densify", "densify", 30000, 4, 1, 1, 803, 601, 12),
    ]


def draw(rng):
    """A case of the same kinds, sizes spread over their logarithm."""
    kind = rng.choice(("render", "views", "train", "batch", "batch", "multi", "autograd", "interval", "densify"))
    log = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    points = log(500, 60000)
    sh = -1 if kind in ("autograd", "interval") else rng.choice((0, 1, 2, 3, 3)) if kind == "multi" else rng.choice(
        (-1, 0, 1, 2, 3, 3))
    views = log(1, 12) if kind in ("views", "batch") else rng.randint(1, 3) if kind == "multi" else 1
    return {"kind": kind, "points": points, "clusters": rng.choice((0, 0, 4, 6, 8)), "sh": sh, "views": views,
            "width": log(96, 1024), "height": log(96, 1024), "tile": rng.choice((8, 12, 12, 16, 16, 32)),
            "loss": rng.choice((0, 1)),
            "adjoint": rng.choice(("undo", "undo", "checkpoint")) if kind in ("batch", "train") else "undo",
            "fwd": 0, "bwd": 0}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=24)
def _mesh(points, clusters):
    """The mesh of a size (built once per process: Delaunay takes seconds); the seeds turn it."""
    rng = np.random.default_rng(points * 31 + clusters)
    p = uniform_points(points, rng) if not clusters else cluster_points(points, rng, clusters, 0.15)
    p = p.astype(np.float32)
    return p.astype(np.float64), delaunay_tets(p)


def _scene(points, clusters, sh, rng):
    p, tets = _mesh(points, clusters)
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    R = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                  [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                  [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])
    M = len(tets)
    f = lambda n, mean, sigma: (rng.standard_normal(n, dtype=np.float32) * sigma + mean).astype(np.float32)  # noqa: E731
    s = {"vertices": (p @ R.T).astype(np.float32).ravel(), "indices": tets.ravel().copy(),
         "densities": np.exp(f(M, 0.0, 1.0)), "color_grads": f(3 * M, 0.0, 0.1)}
    s["circumdata"] = circumspheres(s["vertices"], s["indices"])
    if sh >= 0:
        nc = (sh + 1) ** 2
        c = f((M, 3, nc), 0.0, 0.3)
        c[:, :, 0] = f((M, 3), 0.5, 0.2)
        s |= {"sh": c.ravel(), "sh_degree": sh, "base_colors": np.zeros(3 * M, np.float32)}
    else:
        s["base_colors"] = f(3 * M, 0.5, 0.3)
    return s


def _target(h, w, rng):
    """A smooth image in (0, 1) with grain."""
    yy, xx = np.meshgrid(np.linspace(0, 1, h, dtype=np.float32), np.linspace(0, 1, w, dtype=np.float32), indexing="ij")
    img = np.full((h, w, 3), 0.5, np.float32)
    for _ in range(4):
        a, b = rng.uniform(-9, 9, 2).astype(np.float32)
        img += np.sin(a * xx + b * yy + np.float32(rng.uniform(0, 6)))[..., None] * rng.uniform(0, 0.1, 3).astype(np.float32)
    img += rng.standard_normal((h, w, 3), dtype=np.float32) * np.float32(0.02)
    return np.ascontiguousarray(img)


def _inputs(case, seed):
    """Scenes (one, or several uneven ones for "multi"), cameras and targets of a case, from the seed alone."""
    rng = np.random.default_rng([seed, 77])
    W, H, V = case["width"], case["height"], case["views"]
    parts = [(case["points"], case["clusters"], case["sh"], W, H)]
    if case["kind"] == "multi":
        degs = (case["sh"], 0, 1, 3)
        parts = [(max(400, case["points"] // (i * i + 1)), case["clusters"] if i % 2 == 0 else 0, degs[i],
                  max(64, W * (4 - i) // 4), max(64, H * (i + 2) // 5)) for i in range(4)]
    out = []
    for points, clusters, sh, w, h in parts:
        out.append({"scene": _scene(points, clusters, sh, rng), "w": w, "h": h,
                    "cams": fibonacci_cameras(V, 3.0, 50.0, w, h),
                    "gt": np.stack([_target(h, w, rng) for _ in range(V)]) if case["kind"] not in ("render", "views")
                    else None})
    return out


class _DeviceArray:
    def __init__(self, r, which, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (r.device_buffer(which), False),
                                         "version": 2}


def _view(r, which, n):
    """Zero-copy tensor over one of the renderer's device buffers.  The tensor
    holds the renderer: the buffer lives as long as the renderer does."""
    t = torch.as_tensor(_DeviceArray(r, which, n), device="cuda")
    t.renderer = r
    return t


def _weights(r, n, m, n_sh):
    v = {"vertices": (_lib.BUF_VERTICES, 3 * n), "densities": (_lib.BUF_DENSITIES, m),
         "color_grads": (_lib.BUF_COLOR_GRADS, 3 * m), "d_vertices": (_lib.BUF_D_VERTICES, 3 * n),
         "d_densities": (_lib.BUF_D_DENSITIES, m), "d_color_grads": (_lib.BUF_D_COLOR_GRADS, 3 * m)}
    if n_sh:
        v["sh"] = (_lib.BUF_SH, n_sh)
    return {k: _view(r, *a) for k, a in v.items()}


def _renderer(case, part, **kw):
    s = part["scene"]
    return RMeshRenderer(s["vertices"], s["indices"], s["base_colors"], s["densities"], s["color_grads"],
                         s["circumdata"], part["w"], part["h"], tile_size=case["tile"], sh_coeffs=s.get("sh"),
                         sh_degree=s.get("sh_degree", 0), max_views=case["views"], **kw)


def prepare(case, seed):
    kind, parts = case["kind"], _inputs(case, seed)
    one = parts[0]
    s, cams = one["scene"], one["cams"]
    n, m = len(s["vertices"]) // 3, len(s["densities"])
    st = {"kind": kind, "case": case, "cams": cams, "cam": cams[0]}
    if kind == "multi":
        r = MultiSceneRenderer([dict(p["scene"], width=p["w"], height=p["h"]) for p in parts], tile_size=case["tile"],
                               max_views=case["views"])
        st["nv"] = [case["views"]] * len(parts)
        st["cams"] = [c for p in parts for c in p["cams"]]
        r.set_targets(st["nv"], [p["gt"] for p in parts])
        r.set_graph_mode(True)
        st["weights"] = _weights(r, sum(len(p["scene"]["vertices"]) // 3 for p in parts),
                                 sum(len(p["scene"]["densities"]) for p in parts),
                                 sum(len(p["scene"]["sh"]) for p in parts))
        return st | {"r": r}
    if kind == "autograd":
        mod = RMeshModule(s["vertices"], s["indices"], s["base_colors"], s["densities"], s["color_grads"],
                          s["circumdata"], one["w"], one["h"], tile_size=case["tile"]).cuda()
        return st | {"mod": mod, "gt": torch.from_numpy(one["gt"][0]).cuda(),
                     "cam_t": [torch.from_numpy(c) for c in cams[0]]}
    r = _renderer(case, one)
    if case["fwd"] or case["bwd"]:
        r.set_tuning(case["tile"], case["fwd"], case["bwd"])
    if case["adjoint"] != "undo":
        r.set_adjoint_mode(case["adjoint"])
    st["r"] = r
    if kind == "views":
        st["images"] = _view(r, _lib.BUF_RGBA, case["views"] * one["h"] * one["w"] * 4)
    elif kind in ("train", "batch"):
        st["weights"] = _weights(r, n, m, len(s.get("sh", ())))
        st["lr_sh"] = LR[3] if "sh" in s else 0.0
        if kind == "batch":
            r.set_targets(one["gt"])
            r.set_graph_mode(True)
        else:
            st["gt"] = one["gt"][0]
    elif kind == "interval":
        st["dl"] = _upstream(one)
    elif kind == "densify":
        st["err"] = np.abs(one["gt"][0][..., 0] - 0.5), np.abs(one["gt"][0][..., 1] - 0.5)
        st["err"] = tuple(np.ascontiguousarray(e) for e in st["err"])
    return st


def _upstream(part):
    """An image gradient of a squared loss's size, none on alpha."""
    h, w = part["h"], part["w"]
    dl = np.zeros((h, w, 4), np.float32)
    dl[..., :3] = (part["gt"][0] - np.float32(0.4)) * np.float32(2.0 / (w * h))
    return dl


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "autograd":
        mod = st["mod"]
        mod.zero_grad(set_to_none=True)
        img = mod(*st["cam_t"])
        loss = (img[..., :3] - st["gt"]).square().mean()
        loss.backward()
        return {"image": img.detach(), "loss": loss.detach()} | {"d_" + k: p.grad for k, p in mod.named_parameters()}
    r = st["r"]
    if kind == "render":
        return r.forward_tiled(*st["cam"])
    if kind == "views":
        r.forward_batched(st["cams"], copy_out=False)
        return st["images"]
    if kind == "train":
        loss = r.train_step(*st["cam"], st["gt"], *LR[:3], case["loss"], lr_sh=st["lr_sh"])
        return {"loss": loss} | st["weights"]
    if kind == "batch":
        loss = r.train_step_batched(st["cams"], case["loss"], *LR[:3], lr_sh=st["lr_sh"])
        return {"loss": loss} | st["weights"]
    if kind == "multi":
        loss, per_view = r.train_step(st["nv"], st["cams"], case["loss"], *LR)
        return {"loss": loss, "per_view": per_view} | st["weights"]
    if kind == "interval":
        return r.forward_interval_tiled(*st["cam"]) | r.backward_interval_tiled(st["dl"])
    img, aux = r.forward_tiled(*st["cam"], render_aux=True)
    err, count = r.forward_error(*st["err"])
    return {"image": img, "aux": aux, "tet_err": err, "tet_count": count}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: parameters, images and states read and written once.  Flops: per
    covered (pixel, tet) pair, the slab test, the volume integral and its
    compositing, about 120, and about 220 more for its adjoint; a ray of the
    covered quarter of the image crosses about 3.4 cbrt(points) tets."""
    train = case["kind"] in ("train", "batch", "multi")
    adj = train or case["kind"] in ("autograd", "interval")
    total = {"bytes": 0.0, "flops": 0.0}
    parts = [(case["points"], case["sh"], case["width"], case["height"])]
    if case["kind"] == "multi":
        degs = (case["sh"], 0, 1, 3)
        parts = [(max(400, case["points"] // (i * i + 1)), degs[i], max(64, case["width"] * (4 - i) // 4),
                  max(64, case["height"] * (i + 2) // 5)) for i in range(4)]
    for n, sh, w, h in parts:
        m, px = 6.7 * n, w * h * case["views"]
        col = 3 * (sh + 1) ** 2 if sh >= 0 else 3
        params = 3 * n + 4 * m + (col * m if sh >= 0 else 0)
        b = 4 * (3 * n + 4 * m + 4 * m + m + 3 * m + col * m) + 16 * px
        if train:
            b += 4 * (5 * params) + 4 * (3 * n + 4 * m) + 12 * px  # m, v in and out, weights out, gradients, targets
        elif adj:
            b += 4 * (3 * n + 7 * m) + 12 * px
        if case["kind"] == "interval":
            b += 36 * px
        if case["kind"] == "densify":
            b += 72 * m + 40 * px
        pairs = px * 0.25 * 3.4 * n ** (1 / 3)
        total["bytes"] += b
        total["flops"] += pairs * (120 + (220 if adj else 0))
    return total


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
FACES = ((0, 2, 1, 3), (1, 2, 3, 0), (0, 3, 2, 1), (3, 0, 1, 2))
CHUNK = 40_000_000  # candidate (pixel, tet) pairs looked at together


def _t64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().double()


class _Mesh64:
    """A scene's parameters as float64 leaves."""

    def __init__(self, s, grad):
        self.idx = torch.from_numpy(s["indices"].reshape(-1, 4).astype(np.int64)).cuda()
        self.verts = _t64(s["vertices"]).view(-1, 3).requires_grad_(grad)
        self.dens = _t64(s["densities"]).requires_grad_(grad)
        self.g = _t64(s["color_grads"]).view(-1, 3).requires_grad_(grad)
        self.base = _t64(s["base_colors"]).view(-1, 3).requires_grad_(grad and "sh" not in s)
        self.sh = _t64(s["sh"]).view(len(s["densities"]), 3, -1).requires_grad_(grad) if "sh" in s else None
        self.circ = torch.from_numpy(s["circumdata"].reshape(-1, 4)).cuda()

    def leaves(self):
        return [self.verts, self.dens, self.g, self.base if self.sh is None else self.sh]


def _sh_basis(d, nc):
    x, y, z = d.unbind(-1)
    Y = [torch.full_like(x, 0.5 / math.sqrt(math.pi))]
    if nc > 1:
        c = math.sqrt(3 / (4 * math.pi))
        Y += [-c * y, c * z, -c * x]
    if nc > 4:
        a, b = math.sqrt(15 / (4 * math.pi)), math.sqrt(5 / (16 * math.pi))
        Y += [a * x * y, -a * y * z, b * (2 * z * z - x * x - y * y), -a * x * z, a / 2 * (x * x - y * y)]
    if nc > 9:
        p, q = math.sqrt(35 / (32 * math.pi)), math.sqrt(105 / (4 * math.pi))
        r, t = math.sqrt(21 / (32 * math.pi)), math.sqrt(7 / (16 * math.pi))
        Y += [-p * y * (3 * x * x - y * y), q * x * y * z, -r * y * (4 * z * z - x * x - y * y),
              t * z * (2 * z * z - 3 * x * x - 3 * y * y), -r * x * (4 * z * z - x * x - y * y),
              q / 2 * z * (x * x - y * y), -p * x * (x * x - 3 * y * y)]
    return torch.stack(Y, -1)


def _colors(ms, cam):
    """Per-tet colours seen from cam."""
    if ms.sh is None:
        return ms.base
    v = ms.verts[ms.idx]
    cen = v.mean(1)
    d = cen - cam
    Y = _sh_basis(d / d.norm(dim=-1, keepdim=True), ms.sh.shape[-1])
    x = (ms.sh * Y[:, None, :]).sum(-1) + 0.5 + (ms.g * (v[:, 0] - cen)).sum(-1, keepdim=True)
    return torch.where(x * 10 > 20, x, 0.1 * torch.log1p(torch.exp(torch.clamp(10 * x, max=30.0))))


def _project(ms, cam3, W, H):
    """Clip coordinates, pixel positions and the tets that the renderer bins (its culling rules)."""
    _, vp, _ = cam3
    v = ms.verts[ms.idx]
    P = _t64(vp).view(4, 4).t()
    clip = v @ P[:, :3].t() + P[:, 3]
    w = clip[..., 3]
    ndc = clip[..., :3] / w[..., None]
    lo, hi = ndc.min(1).values, ndc.max(1).values
    ok = (w > 0).all(1) & (hi[:, 0] >= -1) & (lo[:, 0] <= 1) & (hi[:, 1] >= -1) & (lo[:, 1] <= 1) & (lo[:, 2] <= 1)
    ok &= (hi[:, 0] - lo[:, 0]) * W * (hi[:, 1] - lo[:, 1]) * H >= 1
    e = torch.stack([(v[:, a] - v[:, b]).square().sum(-1) for a in range(4) for b in range(a)]).max(0).values
    ok &= ms.dens * e.sqrt() >= 0.01
    pix = torch.stack([(ndc[..., 0] + 1) * 0.5 * W, (1 - ndc[..., 1]) * 0.5 * H], -1)
    return clip, ndc, pix, ok


def _candidates(pix, ok, W, H):
    """Chunks of (tet, x, y): the pixels whose centre lies in a tet's screen box."""
    x0 = (pix[..., 0].min(1).values - 0.5).ceil().clamp(0, W).long()
    x1 = (pix[..., 0].max(1).values - 0.5).floor().clamp(-1, W - 1).long()
    y0 = (pix[..., 1].min(1).values - 0.5).ceil().clamp(0, H).long()
    y1 = (pix[..., 1].max(1).values - 0.5).floor().clamp(-1, H - 1).long()
    nx = (x1 - x0 + 1).clamp(min=0)
    n = torch.where(ok, nx * (y1 - y0 + 1).clamp(min=0), 0)
    t = n.nonzero()[:, 0]
    cut = torch.div(n[t].cumsum(0), CHUNK, rounding_mode="floor")
    for c in range(int(cut[-1]) + 1 if len(t) else 0):
        tc = t[cut == c]
        if not len(tc):
            continue
        k = torch.repeat_interleave(tc, n[tc])
        first = n[tc].cumsum(0) - n[tc]
        j = torch.arange(len(k), device=k.device) - torch.repeat_interleave(first, n[tc])
        yield k, x0[k] + j % nx[k], y0[k] + torch.div(j, nx[k], rounding_mode="floor")


def _rays(cam3, W, H):
    ci = _t64(cam3[2])
    x = (torch.arange(W, device="cuda", dtype=torch.float64) + 0.5 - ci[14]) / ci[12]
    y = (torch.arange(H, device="cuda", dtype=torch.float64) + 0.5 - ci[15]) / ci[13]
    yy, xx = torch.meshgrid(y, x, indexing="ij")
    d = torch.stack([xx, yy, torch.ones_like(xx)], -1)
    scale = d.norm(dim=-1)
    d = d / scale[..., None]
    d = d[..., :1] * ci[0:3] + d[..., 1:2] * ci[4:7] + d[..., 2:] * ci[8:11]
    return (d / d.norm(dim=-1, keepdim=True)).view(-1, 3), scale.view(-1)


def _depth_order(ms, cam3):
    """Rank of every tet, front to back: ascending bits of the float32 power
    distance (the sort key of the tile lists), the later tet first among equals."""
    d = ms.circ[:, :3] - torch.from_numpy(cam3[0]).cuda()
    p = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
    bits = (p - ms.circ[:, 3]).view(torch.int32).long() & 0xFFFFFFFF
    M = len(bits)
    order = torch.sort(bits * M + (M - 1 - torch.arange(M, device="cuda"))).indices
    rank = torch.empty_like(order)
    rank[order] = torch.arange(M, device="cuda")
    return rank


def _planes(ms, cam):
    """Inward face normals n and n . (face vertex - cam), [M, 4, ...]."""
    v = ms.verts[ms.idx]
    n, num = [], []
    for a, b, c, o in FACES:
        q = torch.linalg.cross(v[:, c] - v[:, a], v[:, b] - v[:, a])
        q = torch.where((q * (v[:, o] - v[:, a])).sum(-1, keepdim=True) < 0, -q, q)
        n.append(q)
        num.append((q * (v[:, a] - cam)).sum(-1))
    return torch.stack(n, 1), torch.stack(num, 1)


def _sorted_hits(pixel, tet, rank, more):
    order = torch.sort(pixel * len(rank) + rank[tet]).indices
    return [x[order] for x in (pixel, tet, *more)]


def _slab_hits(ms, cam3, W, H):
    """Covered (pixel, tet) pairs by pixel, front to back, with their entry and exit faces."""
    with torch.no_grad():
        cam = _t64(cam3[0])
        _, _, pix, ok = _project(ms, cam3, W, H)
        n, num = _planes(ms, cam)
        rays, _ = _rays(cam3, W, H)
        got = []
        for k, x, y in _candidates(pix, ok, W, H):
            p = y * W + x
            tmin = torch.full_like(k, -1, dtype=torch.float64).fill_(-math.inf)
            tmax = torch.full_like(tmin, math.inf)
            fa, fb = torch.zeros_like(k), torch.zeros_like(k)
            rd = rays[p]
            for f in range(4):
                den = (n[k, f] * rd).sum(-1)
                t = num[k, f] / den
                a, b = (den > 0) & (t > tmin), (den < 0) & (t < tmax)
                tmin, fa = torch.where(a, t, tmin), torch.where(a, f, fa)
                tmax, fb = torch.where(b, t, tmax), torch.where(b, f, fb)
            h = tmin < tmax
            got.append((p[h], k[h], fa[h], fb[h]))
        if not got:
            z = torch.zeros(0, dtype=torch.long, device="cuda")
            return z, z, z, z
        p, k, fa, fb = (torch.cat(x) for x in zip(*got))
        del got
        return _sorted_hits(p, k, _depth_order(ms, cam3), (fa, fb))


def _integral(od, cs, ce):
    """Premultiplied colour of a slab whose colour runs linearly from cs to ce, and its weights."""
    at = torch.exp(-od)
    ph = torch.where(od < 1e-5, 1 - od / 2 + od * od / 6, -torch.expm1(-od) / od)
    w0, w1 = ph - at, 1 - ph
    return ce * w0[:, None] + cs * w1[:, None], w0, w1, at


def _slab_terms(ms, cam3, hits, rays):
    """od, premultiplied colour, t_min, t_max, w0, transmittance of every hit (differentiable)."""
    p, k, fa, fb = hits
    cam = _t64(cam3[0])
    n, num = _planes(ms, cam)
    n, num = n.reshape(-1, 3), num.reshape(-1)
    rd = rays[p]
    ta = num[4 * k + fa] / (n[4 * k + fa] * rd).sum(-1)
    tb = num[4 * k + fb] / (n[4 * k + fb] * rd).sum(-1)
    base = _colors(ms, cam) + (ms.g * (cam - ms.verts[ms.idx[:, 0]])).sum(-1, keepdim=True)
    slope = (ms.g[k] * rd).sum(-1)
    b = base[k]
    cs, ce = torch.relu(b + (slope * ta)[:, None]), torch.relu(b + (slope * tb)[:, None])
    od = (ms.dens[k] * (tb - ta)).clamp(1e-8, 88.0)
    cp, w0, _, at = _integral(od, cs, ce)
    return od, cp, ta, tb, w0, at


def _before(p, od):
    """Sum of od over the earlier hits of the same pixel."""
    c = od.cumsum(0) - od
    new = torch.ones_like(p, dtype=torch.bool)
    new[1:] = p[1:] != p[:-1]
    first = new.nonzero()[:, 0]
    return c - c[first][new.cumsum(0) - 1]


def _composite(p, od, cp, npx):
    """Image, log T before every hit, which hits count (log T >= -13.8) and each pixel's last log T."""
    before = -_before(p, od)
    live = before >= -13.8
    T = torch.where(live, torch.exp(before), 0.0)
    rgb = torch.zeros(npx, 3, dtype=torch.float64, device="cuda").index_add_(0, p, cp * T[:, None])
    end = torch.zeros(npx, dtype=torch.float64, device="cuda").index_add_(0, p, torch.where(live, -od, 0.0))
    alpha = 1 - torch.exp(end.clamp(min=-88.0))
    return torch.cat([rgb, alpha[:, None]], 1), before, live, T, end


def _backward_sum(p, od, cp, img, live, T, dl, undo):
    """A scalar whose gradient is the renderer's adjoint for the colour gradient dl.

    The adjoint walks a pixel's hits from the back and, in the undo mode,
    rebuilds log T from the image's alpha over all of them; T is held, and the
    hits in front enter through the optical depth alone."""
    if undo:
        with torch.no_grad():
            tot = torch.zeros(len(img), dtype=torch.float64, device="cuda").index_add_(0, p, od)
            left = torch.log((1 - img[:, 3]).clamp(min=1e-20))
            lt = torch.minimum(left[p] + tot[p] - _before(p, od), torch.zeros((), dtype=torch.float64, device="cuda"))
            T = torch.exp(lt)
            live = T >= 1e-6
    c = torch.where(live, _before(p, torch.where(live, od, 0.0)), 0.0)
    w = torch.where(live, T, 0.0) * torch.exp(-(c - c.detach()))
    return ((dl[p] * cp).sum(-1) * w).sum()


def _loss_grad(rgb, gt, loss_type):
    """Loss and d loss / d rgb (mean over pixels of the sum over channels)."""
    d, n = rgb - gt, len(gt)
    return (d.abs().sum() / n, d.sign() / n) if loss_type == 0 else (d.square().sum() / n, 2 * d / n)


def _adam(p, g, lr):
    """A first Adam step."""
    g = torch.nan_to_num(g, nan=0.0).clamp(-1e20, 1e20)
    return p - lr * g / (g.abs() + 1e-8)


def _exact_train(part, loss_type, undo):
    ms, W, H = _Mesh64(part["scene"], True), part["w"], part["h"]
    losses = []
    for cam3, gt in zip(part["cams"], part["gt"]):
        hits = _slab_hits(ms, cam3, W, H)
        od, cp = _slab_terms(ms, cam3, hits, _rays(cam3, W, H)[0])[:2]
        img, _, live, T, _ = _composite(hits[0], od.detach(), cp.detach(), W * H)
        loss, dl = _loss_grad(img[:, :3], _t64(gt).view(-1, 3), loss_type)
        losses.append(float(loss))
        _backward_sum(hits[0], od, cp, img, live, T, dl, undo).backward()
        del od, cp, hits, img, live, T
    return ms, losses


def _exact_weights(ms):
    g = [x.grad if x.grad is not None else torch.zeros_like(x) for x in ms.leaves()]
    out = {"d_vertices": g[0], "d_densities": g[1], "d_color_grads": g[2], "vertices": _adam(ms.verts.detach(), g[0], LR[0]),
           "densities": _adam(ms.dens.detach(), g[1], LR[1]), "color_grads": _adam(ms.g.detach(), g[2], LR[2])}
    if ms.sh is not None:
        out["sh"] = _adam(ms.sh.detach(), g[3], LR[3])
    return {k: v.reshape(-1) for k, v in out.items()}


def _exact_interval(part):
    """Image, depth, distortion and the image's adjoint with the screen geometry held."""
    ms, W, H, cam3 = _Mesh64(part["scene"], True), part["w"], part["h"], part["cams"][0]
    near, far = 0.01, 1000.0
    cam = _t64(cam3[0])
    _, ndc, pix, ok = _project(ms, cam3, W, H)
    pix = pix.detach()
    z = ndc[..., 2]
    off = (ms.g[:, None] * (ms.verts[ms.idx] - cam)).sum(-1)
    base = _colors(ms, cam) + (ms.g * (cam - ms.verts[ms.idx[:, 0]])).sum(-1, keepdim=True)
    M, ar = len(ms.idx), torch.arange(len(ms.idx), device="cuda")
    cross = lambda a, b: a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]  # noqa: E731

    def bary(q, a, b, c):
        v0, v1, v2 = b - a, c - a, q - a
        d00, d01, d11 = (v0 * v0).sum(-1), (v0 * v1).sum(-1), (v1 * v1).sum(-1)
        d20, d21 = (v2 * v0).sum(-1), (v2 * v1).sum(-1)
        det = d00 * d11 - d01 * d01
        inv = torch.where(det.abs() > 1e-10, 1 / det, 0.0)
        b1, b2 = (d11 * d20 - d01 * d21) * inv, (d00 * d21 - d01 * d20) * inv
        return torch.stack([1 - b1 - b2, b1, b2], -1)

    def meet(a1, a2, b1, b2):
        d = cross(a2 - a1, b2 - b1)
        return torch.where(d.abs() < 1e-10, -1.0, cross(b1 - a1, b2 - b1) / d)

    ok = ok & (z.max(1).values - z.min(1).values >= 1e-7) & (ms.dens >= 1e-6)
    # slots 0-3: silhouette points as vertex ids; the centre as weights of two combinations of the vertices
    sil = torch.zeros(M, 4, dtype=torch.long, device="cuda")
    wa, wb = torch.zeros(M, 4, dtype=torch.float64, device="cuda"), torch.zeros(M, 4, dtype=torch.float64, device="cuda")
    inner = torch.full((M,), -1, device="cuda")
    for f in (3, 2, 1, 0):
        a, b, c, q = FACES[f]
        s = torch.stack([cross(pix[:, j] - pix[:, i], pix[:, q] - pix[:, i]) for i, j in ((a, b), (b, c), (c, a))])
        inner = torch.where((s >= 0).all(0) | (s <= 0).all(0), q, inner)
    for q in range(4):
        a, b, c, o = FACES[(q + 1) % 4]
        m = (inner == q).nonzero()[:, 0]
        wt = bary(pix[m, o], pix[m, a], pix[m, b], pix[m, c])
        sil[m] = torch.tensor([a, b, c, a], device="cuda")
        for i, j in enumerate((a, b, c)):
            wa[m, j] = wt[:, i]
        wb[m, o] = 1.0
    quad, left = inner < 0, inner < 0
    for n, (a0, a1, b0, b1) in enumerate(((0, 1, 2, 3), (0, 2, 1, 3), (0, 3, 1, 2), (0, 1, 2, 3))):
        ta = meet(pix[:, a0], pix[:, a1], pix[:, b0], pix[:, b1])
        tb = meet(pix[:, b0], pix[:, b1], pix[:, a0], pix[:, a1])
        m = left if n == 3 else left & (ta > 0) & (ta < 1) & (tb > 0) & (tb < 1)
        left = left & ~m
        m = m.nonzero()[:, 0]
        sil[m] = torch.tensor([a0, b0, a1, b1], device="cuda")
        wa[m, a0], wa[m, a1], wb[m, b0], wb[m, b1] = 1 - ta[m], ta[m], 1 - tb[m], tb[m]
    centre = torch.where(quad[:, None], (wa[..., None] * pix).sum(1), (wb[..., None] * pix).sum(1))
    za, zb = (wa * z).sum(1), (wb * z).sum(1)
    oa, ob = (wa * off).sum(1), (wb * off).sum(1)
    a_first = za <= zb
    cz = torch.stack([torch.minimum(za, zb), torch.maximum(za, zb)], -1)
    co = torch.stack([torch.where(a_first, oa, ob), torch.where(a_first, ob, oa)], -1)
    spix, sz, so = pix[ar[:, None], sil], z.gather(1, sil), off.gather(1, sil)
    rank, (_, scale) = _depth_order(ms, cam3), _rays(cam3, W, H)
    got = []
    with torch.no_grad():
        for k, x, y in _candidates(pix, ok, W, H):
            q = torch.stack([x + 0.5, y + 0.5], -1).double()
            fan = torch.full_like(k, -1)
            for i in (3, 2, 1, 0):
                j = torch.where(quad[k], (i + 1) % 4, (i + 1) % 3)
                a, b, c = spix[k, i], spix[k, j], centre[k]
                d = torch.stack([cross(b - a, q - a), cross(c - b, q - b), cross(a - c, q - c)])
                inside = ~((d < 0).any(0) & (d > 0).any(0))
                fan = torch.where(inside & (quad[k] | (i < 3)), i, fan)
            h = fan >= 0
            got.append(((y * W + x)[h], k[h], fan[h]))
        p, k, i = (torch.cat(x) for x in zip(*got))
        p, k, i = _sorted_hits(p, k, rank, (i,))
        j = torch.where(quad[k], (i + 1) % 4, (i + 1) % 3)
        q = torch.stack([p % W + 0.5, torch.div(p, W, rounding_mode="floor") + 0.5], -1).double()
        bc = bary(q, spix[k, i], spix[k, j], centre[k])
    at = lambda s, c: (bc[:, 0] * s[k, i] + bc[:, 1] * s[k, j])[:, None] + bc[:, 2:] * c[k]  # noqa: E731
    lin = near * far / (far - at(sz, cz).clamp(0, 1) * (far - near))
    o = at(so, co)
    zf, zb_ = lin[:, 0], lin[:, 1]
    rs = scale[p]
    od = (ms.dens[k] * (zb_ - zf).abs() * rs).clamp(1e-8, 88.0)
    cp, w0, w1, _ = _integral(od, torch.relu(base[k] + o[:, :1]), torch.relu(base[k] + o[:, 1:]))
    img, before, live, T, _ = _composite(p, od.detach(), cp.detach(), W * H)
    _backward_sum(p, od, cp, img, live, T, _t64(_upstream(part)).view(-1, 4)[:, :3], True).backward()
    with torch.no_grad():
        add = lambda v: torch.zeros(W * H, dtype=torch.float64, device="cuda").index_add_(0, p, v)  # noqa: E731
        dens, enter, leave = ms.dens[k], zf * rs, zb_ * rs
        u = dens * (leave - enter)
        en = torch.exp(-u)
        m0 = T * (1 - en).clamp(min=0)
        m1 = T * (enter * (1 - en).clamp(min=0) + (1 - (1 + u) * en) / dens)
        m2 = T * T * (1 - 2 * u * en - en * en) / dens
        dist = torch.stack([add(2 * m1 * _before(p, m0)), add(2 * m0 * _before(p, m1)), add(m0), add(m1), add(m2)], -1)
        xyzd = torch.zeros(W * H, 4, dtype=torch.float64, device="cuda")
        xyzd[:, 3] = add(T * (w0 * zb_ + w1 * zf))
    return {"image": img.view(H, W, 4), "xyzd": xyzd.view(H, W, 4), "distortion": dist.view(H, W, 5),
            "d_vertices": ms.verts.grad.reshape(-1), "d_densities": ms.dens.grad,
            "d_base_colors": ms.base.grad.reshape(-1), "d_color_grads": ms.g.grad.reshape(-1),
            "d_vertex_normals": torch.zeros_like(ms.verts).reshape(-1)}


def _exact_densify(part):
    ms, W, H, cam3 = _Mesh64(part["scene"], False), part["w"], part["h"], part["cams"][0]
    hits, rays, cam = _slab_hits(ms, cam3, W, H), _rays(cam3, W, H)[0], _t64(cam3[0])
    p, k, fa, _ = hits
    od, cp, ta, tb, w0, at = _slab_terms(ms, cam3, hits, rays)
    img, before, live, T, _ = _composite(p, od, cp, W * H)
    n = _planes(ms, cam)[0][k, fa]
    wt, mid = T * (1 - at), (ta + tb) / 2
    wc = wt * mid
    xlog = lambda x: torch.where(x > 1e-20, x * torch.log(x.clamp(min=1e-300)), 0.0)  # noqa: E731
    depth = T * (w0 * tb + (1 - (w0 + at)) * ta)
    cols = [*(-n / n.norm(dim=-1, keepdim=True) * wt[:, None]).unbind(-1), depth, wt, xlog(wt), wc, xlog(wc)]
    aux = torch.zeros(W * H, 8, dtype=torch.float64, device="cuda").index_add_(0, p, torch.stack(cols, -1))
    gt = part["gt"][0]
    pe, se = (_t64(np.abs(gt[..., c] - 0.5)).view(-1)[p] for c in (0, 1))
    tv = torch.where(before >= -5.5, T * od, 0.0)
    en, ex = cam + rays[p] * ta[:, None], cam + rays[p] * tb[:, None]
    cen = ms.verts[ms.idx].mean(1)[k]
    z = torch.zeros_like(tv)
    cols = [tv, tv * pe, tv * pe * pe, z, z, tv * se, *(en * tv[:, None]).unbind(-1), *(ex * tv[:, None]).unbind(-1), tv,
            *(cen * tv[:, None]).unbind(-1)]
    err = torch.zeros(len(ms.idx), 16, dtype=torch.float64, device="cuda").index_add_(0, k, torch.stack(cols, -1))
    return {"image": img.view(H, W, 4), "aux": aux.view(H, W, 8), "tet_err": err, "tet_count": None}


def exact(case, seed):
    kind, parts = case["kind"], _inputs(case, seed)
    one = parts[0]
    W, H = one["w"], one["h"]
    if kind in ("render", "views"):
        ms, out = _Mesh64(one["scene"], False), []
        for cam3 in one["cams"]:
            hits = _slab_hits(ms, cam3, W, H)
            od, cp = _slab_terms(ms, cam3, hits, _rays(cam3, W, H)[0])[:2]
            out.append(_composite(hits[0], od, cp, W * H)[0])
        return out[0].view(H, W, 4) if kind == "render" else torch.cat(out).reshape(-1)
    if kind in ("train", "batch"):
        ms, losses = _exact_train(one, case["loss"], case["adjoint"] == "undo")
        return {"loss": float(np.mean(losses))} | _exact_weights(ms)
    if kind == "multi":
        # the renderer keeps its scenes' arrays one after another, by SH degree
        got = [_exact_train(p, case["loss"], True) for p in parts]
        order = sorted(range(len(parts)), key=lambda i: parts[i]["scene"]["sh_degree"])
        w = [_exact_weights(got[i][0]) for i in order]
        per_view = np.array([x for _, losses in got for x in losses])
        return {"loss": float(per_view.mean()), "per_view": per_view} | {k: torch.cat([x[k] for x in w]) for k in w[0]}
    if kind == "autograd":
        ms, cam3 = _Mesh64(one["scene"], True), one["cams"][0]
        hits = _slab_hits(ms, cam3, W, H)
        od, cp = _slab_terms(ms, cam3, hits, _rays(cam3, W, H)[0])[:2]
        img, _, live, T, _ = _composite(hits[0], od.detach(), cp.detach(), W * H)
        d = img[:, :3] - _t64(one["gt"][0]).view(-1, 3)
        _backward_sum(hits[0], od, cp, img, live, T, 2 * d / d.numel(), True).backward()
        return {"image": img.view(H, W, 4), "loss": float(d.square().mean()), "d_vertices": ms.verts.grad.reshape(-1),
                "d_base_colors": ms.base.grad.reshape(-1), "d_densities": ms.dens.grad,
                "d_color_grads": ms.g.grad.reshape(-1)}
    return _exact_interval(one) if kind == "interval" else _exact_densify(one)
