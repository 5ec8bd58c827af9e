"""The work that programs give this library, as cases whose time can be measured.

A case names a ``kind`` and its sizes:

* ``exact``  one frame summed over all AVPLs (``Gather.run`` with
             ``useLightCuts = 0``): reference images and small scenes;
* ``sa``     one frame of the progressive renderer with the reference's default
             settings (solid-angle light cut, clustered disk antiradiance),
             added to the accumulation image and normalised;
* ``cut``    one frame of the error-bound light cut with moment estimates and
             clustered cone antiradiance over an LBVH rebuilt for the frame;
* ``points`` a ``SimpleBvh`` build over points, ``avpls`` an ``AvplBvh`` build
             over AVPLs with position and normal codes;
* ``trace``  the scene side of a frame: a G-buffer cast and AVPLs shot into
             the triangle scene;
* ``batch``  one graph launch that renders several uneven views.

Scenes come from ``antiradiancecuts_amd.scene`` with the case's sizes and the
seed.  Outputs are the library's own device buffers.
"""
import ctypes
import math

import numpy as np
import torch

from antiradiancecuts_amd import ffi, scene
from antiradiancecuts_amd.runtime import (CONE_10DEG, Batch, Bvh, Context, DeviceAvpls, Gather, TraceScene,
                                          default_params, device_array)

MODELS = {"disk": 0, "cone": 1}  # ARC_ANTIRAD_DISK, ARC_ANTIRAD_CONE
MAX_EXACT_PAIRS = 3e10            # (pixel, AVPL) pairs that exact() sums


def listed():
    return [
        # a thumbnail while a scene is edited: launches and the host path are what it waits for
        {"name": "exact_thumbnail", "kind": "exact", "width": 64, "height": 48, "avpls": 500, "model": "disk",
         "phong": False},
        # the reference image of the Cornell box, every pixel with every AVPL
        {"name": "exact_cornell_256", "kind": "exact", "width": 256, "height": 256, "avpls": 4096, "model": "cone",
         "phong": False},
        # a reference image of glossy materials at an odd window size
        {"name": "exact_phong_ragged", "kind": "exact", "width": 331, "height": 247, "avpls": 3001, "model": "disk",
         "phong": True},
        # the interactive renderer as configured out of the box, at 720p
        {"name": "frame_default_720p", "kind": "sa", "width": 1280, "height": 720, "avpls": 65536, "tris": 20000},
        # a small preview window of the error-bound renderer
        {"name": "cut_preview", "kind": "cut", "width": 200, "height": 120, "avpls": 20000, "tris": 20000,
         "bound": 0.01, "floor": 0.0, "count": 16},
        # the setting within 1e-3 of the exact image, at an odd window size
        {"name": "cut_accurate_ragged", "kind": "cut", "width": 1283, "height": 719, "avpls": 250001, "tris": 100000,
         "bound": 0.0045, "floor": 4.0, "count": 128},
        # the headline frame: 1080p, a million AVPLs, the LBVH rebuilt
        {"name": "cut_1080p_1m", "kind": "cut", "width": 1920, "height": 1080, "avpls": 1000000, "tris": 200000,
         "bound": 0.01, "floor": 0.0, "count": 16},
        # a tree over a handful of points: launch latency
        {"name": "bvh_points_1k", "kind": "points", "n": 1000},
        # the LBVH alone at its full size
        {"name": "bvh_points_1m", "kind": "points", "n": 1000000},
        # an AVPL tree that considers normals, one leaf short of a power of two
        {"name": "bvh_avpls_131071", "kind": "avpls", "n": 131071},
        # a camera move and a new light sample: G-buffer cast and AVPL paths
        {"name": "trace_720p_100k", "kind": "trace", "width": 1280, "height": 720, "paths": 100000, "tris": 100000},
        # offline rendering of several uneven views in one launch
        {"name": "batch_6_views", "kind": "batch", "views": 6, "max_width": 960, "max_height": 540,
         "max_avpls": 250000, "tris": 20000, "bound": 0.01, "floor": 0.0, "count": 16, "shape_seed": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["exact", "sa", "cut", "cut", "points", "avpls", "trace", "batch"])
    if kind == "exact":
        return {"kind": kind, "width": _log_int(rng, 48, 400), "height": _log_int(rng, 32, 300),
                "avpls": _log_int(rng, 100, 5000), "model": rng.choice(["disk", "cone"]),
                "phong": rng.random() < 0.3}
    if kind == "sa":
        return {"kind": kind, "width": _log_int(rng, 160, 1400), "height": _log_int(rng, 120, 800),
                "avpls": _log_int(rng, 1000, 100000), "tris": _log_int(rng, 1000, 30000)}
    if kind == "cut":
        setting = rng.choice([(0.01, 0.0, 16), (0.0045, 4.0, 128), (0.01, 4.0, 64), (0.01, 0.0, 128)])
        w, h = _log_int(rng, 96, 1400), _log_int(rng, 64, 800)
        return {"kind": kind, "width": w, "height": h, "avpls": _log_int(rng, 4000, 300000),
                "tris": _log_int(rng, 4000, 100000), "bound": setting[0], "floor": setting[1], "count": setting[2]}
    if kind == "points":
        return {"kind": kind, "n": _log_int(rng, 50, 1000000)}
    if kind == "avpls":
        return {"kind": kind, "n": _log_int(rng, 50, 300000)}
    if kind == "trace":
        return {"kind": kind, "width": _log_int(rng, 160, 1280), "height": _log_int(rng, 90, 720),
                "paths": _log_int(rng, 500, 100000), "tris": _log_int(rng, 1000, 100000)}
    return {"kind": kind, "views": rng.randint(2, 6), "max_width": _log_int(rng, 256, 960),
            "max_height": _log_int(rng, 192, 540), "max_avpls": _log_int(rng, 16000, 250000),
            "tris": _log_int(rng, 4000, 20000), "bound": 0.01, "floor": 0.0, "count": 16,
            "shape_seed": rng.randint(0, 10 ** 6)}


# ------------------------------------------------------------- inputs --
def _view_sizes(case):
    r = np.random.RandomState(case["shape_seed"])
    out = []
    for _ in range(case["views"]):
        w = int(r.randint(128, case["max_width"] + 1))
        h = int(r.randint(96, case["max_height"] + 1))
        n = int(round(math.exp(r.uniform(math.log(8000), math.log(case["max_avpls"])))))
        out.append((w, h, n))
    return out


def _scene(case, seed):
    if case["kind"] == "exact":
        sc = scene.cornell_256(seed=seed, width=case["width"], height=case["height"], num_avpls=case["avpls"])
        if case["phong"]:  # every other material glossy
            sc.materials[::2, 6:9] = [0.3, 0.25, 0.2]
            sc.materials[::2, 9] = 12.0
        return sc
    return scene.clutter_1080p(seed=seed, width=case["width"], height=case["height"], num_avpls=case["avpls"],
                               num_tris=case["tris"])


def _params(case):
    if case["kind"] == "exact":
        return default_params(useLightCuts=0, antiradianceMode=0, antiradianceModel=MODELS[case["model"]],
                              coneHalfAngle=CONE_10DEG)
    if case["kind"] == "sa":
        return default_params()
    return default_params(cutMode=1, cutEstimator=1, cutCriterion=0, cutPerTile=1, errorBound=case["bound"],
                          cutImageFloor=case["floor"], cutExactCount=case["count"], antiradianceModel=1,
                          coneHalfAngle=CONE_10DEG)


def _gather(ctx, sc):
    g = Gather(ctx, sc.width, sc.height, sc.materials)
    g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), device_array(sc.albedo4))
    return g


def prepare(case, seed):
    kind = case["kind"]
    ctx = Context()
    st = {"kind": kind, "ctx": ctx, "seed": seed}
    if kind == "points":
        st["pos"] = device_array(scene.points(case["n"], seed=seed))
        st["bvh"] = Bvh(ctx)
    elif kind == "avpls":
        sc = scene.clutter_1080p(seed=seed, width=8, height=8, num_avpls=case["n"], num_tris=2000)
        st["avpls"] = DeviceAvpls.from_scene(sc)
        st["bvh"] = Bvh(ctx, consider_normals=True)
    elif kind == "trace":
        d = scene.desc(seed, case["width"], case["height"], 16, 1, 4, 1e-3, 10.0, True, 0.3, False, case["tris"],
                       1e-4, 1e-2)
        ts = scene.triangle_scene(d)
        st["trace"] = TraceScene(ctx, ts)
        st["paths"], st["size"] = case["paths"], (case["width"], case["height"])
        cam = np.random.RandomState(seed % (1 << 31)).uniform(0.3, 0.7, 3)
        st["cam"] = (cam, np.array([0.2, -0.1, -1.0]), np.array([0.0, 1.0, 0.0]))
        # the program's own AVPL arrays, which the shots of its frames go to (about 3.3 AVPLs per path;
        # the shooter's arrays last until its next call)
        cap = 8 * case["paths"] + 256
        st["own"] = {k: torch.zeros((cap, 3), device="cuda") for k in ("pos", "nrm", "dir", "rad", "anti")}
        st["own"].update({k: torch.zeros(cap, dtype=torch.int32, device="cuda") for k in ("mat", "bounce")})
    elif kind == "batch":
        batch = Batch(ctx, lanes=4)
        views, keep = [], []
        for k, (w, h, n) in enumerate(_view_sizes(case)):
            sc = scene.clutter_1080p(seed=seed + 1000 * k, width=w, height=h, num_avpls=n, num_tris=case["tris"])
            g = _gather(batch.lane(k), sc)
            views.append((g, DeviceAvpls.from_scene(sc), sc.cam, sc.extent, _params(case)))
            keep.append(g)
        batch.capture(views)
        st["batch"], st["views"], st["gathers"] = batch, views, keep
    else:
        sc = _scene(case, seed)
        st["gather"] = _gather(ctx, sc)
        st["avpls"] = DeviceAvpls.from_scene(sc)
        st["cam"], st["extent"], st["params"] = sc.cam, sc.extent, _params(case)
        if kind == "sa":
            st["accum"] = torch.zeros_like(st["gather"].result)
            st["image"] = torch.zeros_like(st["gather"].result)
            st["frames"] = 0
    return st


# ---------------------------------------------------------------- run --
class _Borrowed:
    def __init__(self, ptr, shape, kind):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (ptr, False), "version": 2}


def _tensors(state, arrays):
    """The library's device arrays as tensors; made anew when the library has moved an array."""
    key = tuple((p, shape) for p, shape, _ in arrays.values())
    if state.get("key") != key:
        state["tensors"] = {k: torch.as_tensor(_Borrowed(p, shape, kind), device="cuda")
                            for k, (p, shape, kind) in arrays.items()}
        state["key"] = key
    return dict(state["tensors"])


def _tree(state):
    b = state["bvh"]
    p, d, nd = ffi.arc_bvh_param(), ffi.arc_bvh_data(), ffi.arc_avpl_node_data()
    lib = b.lib
    ffi.check(lib.arc_bvh_get_param(b.h, ctypes.byref(p)), "arc_bvh_get_param", b.ctx.h)
    ffi.check(lib.arc_bvh_get_data(b.h, ctypes.byref(d)), "arc_bvh_get_data", b.ctx.h)
    n = p.numLeafs
    arrays = {"codes": (d.morton, (n,), "<i4"), "perm": (d.perm, (n,), "<i4"), "nodes": (p.nodes, (n - 1, 9), "<i4"),
              "parents": (d.parents, (2 * n - 1,), "<i4"), "ranges": (d.ranges, (n - 1, 2), "<i4"),
              "positions": (p.positions, (n, 3), "<f4")}
    if state["kind"] == "avpls":
        ffi.check(lib.arc_bvh_get_node_data(b.h, ctypes.byref(nd)), "arc_bvh_get_node_data", b.ctx.h)
        s = 2 * n - 1
        arrays.update(size=(nd.size, (s,), "<i4"), mat=(nd.materialIndex, (s,), "<i4"),
                      node_pos=(nd.position, (s, 3), "<f4"), node_nrm=(nd.normal, (s, 3), "<f4"),
                      node_rad=(nd.incRadiance, (s, 3), "<f4"), node_dir=(nd.incDirection, (s, 3), "<f4"))
    return _tensors(state, arrays)


def run(state):
    kind = state["kind"]
    if kind == "points":
        state["bvh"].build_points(state["pos"])
        return _tree(state)
    if kind == "avpls":
        state["bvh"].build_avpls(state["avpls"], seed=5489)
        return _tree(state)
    if kind == "trace":
        cam, fwd, up = state["cam"]
        w, h = state["size"]
        pos4, nrm4 = state["trace"].gbuffer(cam, fwd, up, 1.0, w, h)
        s = state["trace"].shoot(state["paths"], state["seed"]).struct
        n = s.numAvpls
        shot = _tensors(state, {"pos": (s.position, (n, 3), "<f4"), "nrm": (s.normal, (n, 3), "<f4"),
                                "dir": (s.incDirection, (n, 3), "<f4"), "rad": (s.incRadiance, (n, 3), "<f4"),
                                "anti": (s.antiradiance, (n, 3), "<f4"), "mat": (s.materialIndex, (n,), "<i4"),
                                "bounce": (s.bounce, (n,), "<i4")})
        for k, v in shot.items():
            state["own"][k][:n].copy_(v)
        return {"avpls": state["own"], "count": n, "pos4": pos4, "nrm4": nrm4}
    if kind == "batch":
        state["batch"].launch()
        return [(g.result, g.radiance, g.antiradiance) for g in state["gathers"]]
    g = state["gather"]
    g.run(state["avpls"], state["cam"], state["extent"], state["params"])
    out = {"result": g.result, "radiance": g.radiance, "antiradiance": g.antiradiance}
    if kind == "sa":  # Renderer::Add and Renderer::Normalize of the progressive image
        state["frames"] += 1
        npix, h, p = g.width * g.height, state["ctx"].h, ctypes.c_void_p
        lib = state["ctx"].lib
        ffi.check(lib.arc_image_accumulate(h, p(state["accum"].data_ptr()), p(g.result.data_ptr()), npix),
                  "arc_image_accumulate", h)
        ffi.check(lib.arc_image_normalize(h, p(state["image"].data_ptr()), p(state["accum"].data_ptr()), npix,
                                          state["frames"]), "arc_image_normalize", h)
        out["image"] = state["image"]
    return out


# --------------------------------------------------------------- work --
def work(case):
    """Inputs read once and outputs written once; for the exact sums the pairs' operations."""
    kind = case["kind"]
    if kind == "points":
        return {"bytes": 80 * case["n"], "flops": 0}
    if kind == "avpls":
        return {"bytes": 276 * case["n"], "flops": 0}
    if kind == "trace":
        # a G-buffer record per pixel, an AVPL per path and bounce (about 3.3 with roulette at 0.8),
        # each triangle once
        return {"bytes": 32 * case["width"] * case["height"] + 68 * 3.3 * case["paths"] + 64 * 2 * case["tris"],
                "flops": 0}
    if kind == "batch":
        return {"bytes": sum(96 * w * h + 68 * n for w, h, n in _view_sizes(case)), "flops": 0}
    npix, n = case["width"] * case["height"], case["avpls"]
    b = {"bytes": 96 * npix + 68 * n, "flops": 0}
    if kind == "exact":
        b["flops"] = (31 + (33 if case["model"] == "cone" else 37)) * npix * n
    elif kind == "sa":
        b["bytes"] += 64 * npix  # the accumulation image read and written, the frame read, the image written
    return b


# -------------------------------------------------------------- exact --
def _dot(a, b):
    return (a * b).sum(-1)


def _unit(a):
    return a / a.norm(dim=-1, keepdim=True)


ONE_OVER_PI = 0.318309886


def _lobe(mirror_cos, spec, expo):
    c = mirror_cos.clamp_min(0.0)
    return (0.5 * ONE_OVER_PI * (expo + 2.0) * c ** expo).unsqueeze(-1) * spec


def _sums(sc, radiance, anti, model):
    """Radiance and antiradiance of every pixel over all AVPLs in 64 bits (either may be left out)."""
    dev = "cuda"
    D = lambda a: torch.from_numpy(np.asarray(a)).to(dev, torch.float64)  # noqa: E731
    pos, nrm, alb = D(sc.pos4[:, :3]), D(sc.nrm4[:, :3]), D(sc.albedo4[:, :3])
    mats = D(sc.materials)
    pm = mats[torch.from_numpy(sc.nrm4[:, 3].astype(np.int64)).to(dev)]
    pspec, pexp = pm[:, 6:9], pm[:, 9]
    cam = D(sc.cam)
    wo = _unit(cam - pos)
    nh = _unit(nrm)
    npix = pos.shape[0]
    R = torch.zeros(npix, 3, device=dev, dtype=torch.float64)
    A = torch.zeros_like(R)
    am = mats[torch.from_numpy(sc.avpl_mat.astype(np.int64)).to(dev)]
    glossy = bool((mats[:, 6:9].abs().sum() > 0).item())
    radius = float(np.float32(2.0) * np.float32(sc.extent) / np.float32(100.0))
    cos_half = math.cos(float(np.float32(CONE_10DEG)))
    n = sc.num_avpls
    some = np.abs(sc.avpl_anti).sum(1) != 0
    lit = np.abs(sc.avpl_rad).sum(1) != 0
    step = max(1, int(2e7 // npix))

    def pixel_brdf(d):  # d: unit, pixel -> AVPL
        b = ONE_OVER_PI * alb.unsqueeze(1)
        if not glossy:
            return b
        mirror = 2.0 * nrm.unsqueeze(1) * _dot(nrm.unsqueeze(1), d).unsqueeze(-1) - d
        return b + _lobe(_dot(mirror, wo.unsqueeze(1)), pspec.unsqueeze(1), pexp.unsqueeze(1)) * \
            (pspec.norm(dim=-1) > 0).view(-1, 1, 1)

    def chunks(mask):
        ids = np.nonzero(mask)[0]
        for k in range(0, len(ids), step):
            yield torch.from_numpy(ids[k:k + step]).to(dev)

    P, N, W = D(sc.avpl_pos), D(sc.avpl_nrm), D(sc.avpl_dir)
    if radiance:
        L = D(sc.avpl_rad)
        for i in chunks(lit):
            d = P[i].unsqueeze(0) - pos.unsqueeze(1)
            dd = _dot(d, d)
            u = d / dd.sqrt().unsqueeze(-1)
            c1 = _dot(nh.unsqueeze(1), u).clamp(0, 1)
            c2 = (-_dot(_unit(N[i]).unsqueeze(0), u)).clamp(0, 1)
            fl = (ONE_OVER_PI * am[i, 3:6]).unsqueeze(0)
            if glossy:
                m = W[i] - 2.0 * N[i] * _dot(N[i], W[i]).unsqueeze(-1)
                fl = fl + _lobe(_dot(m.unsqueeze(0), -u), am[i, 6:9].unsqueeze(0), am[i, 9].unsqueeze(0)) * \
                    (am[i, 6:9].norm(dim=-1) > 0).view(1, -1, 1)
            fl = torch.where((W[i].norm(dim=-1) == 0).view(1, -1, 1), torch.ones_like(fl), fl)
            w = L[i].unsqueeze(0) * fl
            if glossy:
                R += ((c1 * c2 / dd).unsqueeze(-1) * w * pixel_brdf(u)).sum(1)
            else:
                R += ((c1 * c2 / dd) @ w[0]) * (ONE_OVER_PI * alb)
    if anti:
        V = D(sc.avpl_anti)
        for i in chunks(some):
            d = P[i].unsqueeze(0) - pos.unsqueeze(1)
            dd = _dot(d, d)
            u = d / dd.sqrt().unsqueeze(-1)
            w = W[i].unsqueeze(0)
            if model == "cone":
                c = -_dot(u, _unit(W[i]).unsqueeze(0))
                cp = _dot(nrm.unsqueeze(1), u)
                g = torch.where((c > 0.001) & (cp > 0.001) & (c > cos_half), cp / dd, torch.zeros_like(c))
            else:
                den = _dot(w, nrm.unsqueeze(1))
                t = -_dot(d, nrm.unsqueeze(1)) / den
                hit = d + t.unsqueeze(-1) * _unit(W[i]).unsqueeze(0)
                ok = (den < 0) & (t > 0) & (hit.norm(dim=-1) < radius) & (_dot(-u, N[i].unsqueeze(0)) < 0)
                g = ok.to(torch.float64) / (3.14159265 * radius * radius)
            if glossy:
                A += (g.unsqueeze(-1) * V[i].unsqueeze(0) * pixel_brdf(u)).sum(1)
            else:
                A += (g @ V[i]) * (ONE_OVER_PI * alb)
    return R, A


def _image(rgb, w):
    return torch.cat([rgb, torch.full_like(rgb[:, :1], w)], 1)


def exact(case, seed):
    if case["kind"] not in ("exact", "sa", "cut"):
        return None  # trees are whole numbers and copies; paths and views are compared as they are
    pairs = case["width"] * case["height"] * case["avpls"]
    sa = case["kind"] == "sa"
    # (the antiradiance alone: 30 % of the AVPLs carry it)
    if pairs * (0.3 if sa else 1.0) > MAX_EXACT_PAIRS:
        return None
    sc = _scene(case, seed)
    model = case.get("model", "disk" if sa else "cone")
    R, A = _sums(sc, not sa, True, model)
    if sa:  # the solid-angle cut is a random estimate: it has no 64-bit value
        return {"result": None, "radiance": None, "antiradiance": _image(A, 1.0), "image": None}
    return {"result": _image(R - A, 0.0), "radiance": _image(R, 1.0), "antiradiance": _image(A, 1.0)}
