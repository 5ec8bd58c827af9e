"""The moment cut's decisions against a node-by-node walk on the CPU.

The cut of an 8x8 tile is depth first, the lower child first: a node behind
every pixel's tangent plane is dropped, a node of at most cutExactCount AVPLs
is summed exactly, any other is refined when some pixel's bound is above its
threshold, unless the nodes before it have used cutBudget up.  The kernels
decide 64 nodes at a time and meet the budget subtree by subtree; the walk
here takes the device's tree and records and counts what they must count.

FP32 rounding may turn a decision whose bound lies on its threshold: one in
about 1e6 decisions, so at most a few per scene, each moving the counts by one
subtree; the counts are held to 0.5 %.
"""
import numpy as np
import pytest

from antiradiancecuts_amd import ffi
from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import DeviceAvpls, Gather, default_params, device_array

pytestmark = pytest.mark.gpu

f4 = np.float32


def params(**kw):
    base = dict(useLightCuts=1, cutMode=ffi.ARC_CUT_ERROR_BOUND, cutPerTile=1, cutEstimator=ffi.ARC_ESTIMATOR_MOMENTS,
                cutCriterion=ffi.ARC_CRITERION_BOUND, cutImageFloor=0.0, antiradianceModel=ffi.ARC_ANTIRAD_CONE)
    base.update(kw)
    return default_params(**base)


def estimates(nodes, cent, n, pos, nrm, depth=6):
    """The pixel thresholds' estimate: the cut made of the nodes at `depth`."""
    front = [-1]
    for _ in range(depth):
        front = [c for v in front for c in ((nodes[-(v + 1)]["left"], nodes[-(v + 1)]["right"]) if v < 0 else (v,))]
    e = np.zeros(len(pos), np.float64)
    for v in front:
        r = cent[v if v >= 0 else n - (v + 1)].astype(np.float64)
        d = r[0, :3] - pos
        dd = (d * d).sum(1)
        inv = 1 / np.sqrt(dd)
        c1 = np.clip((nrm * d).sum(1) * inv, 0, 1)
        c2 = np.clip(r[1, 3] + np.maximum(-(d @ r[1, :3]) * inv, 0), 0, 1)
        e += r[0, 3] * c1 * c2 * inv * inv
    return e


def walk(nodes, mom, nrm_leaf, P, N, thr, live, delta, exact_count, budget):
    """(tested, visited, kept, exact leaves, budget hits) of one tile."""
    first, count = mom[:, 1, 1].view(np.int32), mom[:, 1, 2].view(np.int32)
    lo, hi = P[live].min(0), P[live].max(0)
    tested = visited = kept = exact = hits = 0
    stack = [-1]
    while stack:
        v = stack.pop()
        if v >= 0:
            exact += 1
            continue
        k = -(v + 1)
        b = nodes[k]
        bl, bh = b["bbMin"], b["bbMax"]
        ex = np.maximum(np.maximum(bl - P, P - bh), 0)
        d2 = np.maximum((ex * ex).sum(1), f4(delta * delta))
        hmax = (N * np.where(N > 0, bh - P, bl - P)).sum(1)
        bound = mom[k, 0, 3] * np.clip(hmax / np.sqrt(d2), 0, 1) / d2
        if not (bound > 0).any():
            continue
        if count[k] <= exact_count:
            exact += int(count[k])
            continue
        tested += 1
        if (bound > thr).any():
            if kept + exact >= budget:
                hits += 1
            else:
                visited += 1
                stack += [int(b["right"]), int(b["left"])]
                continue
        # a kept node whose AVPLs all face away from the tile adds nothing and is not counted
        nn = nrm_leaf[first[k]:first[k] + count[k]]
        nl, nh = nn.min(0), nn.max(0)
        vl, vh = lo - bh, hi - bl
        kept += int(np.maximum(np.maximum(nl * vl, nl * vh), np.maximum(nh * vl, nh * vh)).sum() > -1e-5)
    return tested, visited, kept, exact, hits


@pytest.mark.parametrize("w,h,n,count,bound,budget", [
    (24, 16, 40_000, 16, 1e-4, 20_000),   # tiles that reach their budget among tiles that do not
    (21, 13, 40_000, 128, 1e-4, 20_000),  # ragged tiles, larger exact nodes
    (19, 11, 30_000, 0, 1e-3, 9_000),     # down to single leaves
    (21, 13, 6_000, 16, 1e-3, 300),       # a small budget: the serial cut
    (16, 8, 2, 16, 1e-2, 65_536),         # the smallest tree
    (24, 16, 40_000, 16, 1e-3, 65_536),   # no tile reaches its budget
])
def test_counts_equal_the_serial_walk(gpu_ctx, w, h, n, count, bound, budget):
    print(f"[budget] {w}x{h} n={n} exact<={count} bound {bound:g} budget {budget}", flush=True)
    sc = S.clutter_1080p(seed=11, width=w, height=h, num_avpls=n, num_tris=4000)
    g = Gather(gpu_ctx, w, h, sc.materials)
    g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), device_array(sc.albedo4))
    av = DeviceAvpls.from_scene(sc)
    st = g.run(av, sc.cam, sc.extent, params(errorBound=bound, cutExactCount=count, cutBudget=budget),
               ffi.ARC_RUN_COUNTERS)
    gpu_ctx.sync()
    rad = g.radiance[:, :3].cpu().numpy()
    assert np.isfinite(rad).all()
    tree, cent, mom = g.bvh_to_host(), g.cut_records(ffi.ARC_RECORDS_CENTROID), g.cut_records(ffi.ARC_RECORDS_MOMENTS)
    g.close()
    pos, nrm = sc.pos4[:, :3], sc.nrm4[:, :3] / np.linalg.norm(sc.nrm4[:, :3], axis=1, keepdims=True)
    thr = np.maximum(bound * estimates(tree["nodes"], cent, n, pos, nrm), 1e-30)
    want = np.zeros(5)
    for ty in range((h + 7) // 8):
        for tx in range((w + 7) // 8):
            y, x = [a.ravel() for a in np.mgrid[8 * ty:8 * ty + 8, 8 * tx:8 * tx + 8]]
            live = (x < w) & (y < h)
            q = np.where(live, y * w + x, 0)  # a lane outside the image stands at pixel 0 and asks for nothing
            r = walk(tree["nodes"], mom, cent[:n, 1, :3], pos[q], nrm[q].astype(f4), np.where(live, thr[q], np.inf),
                     live, 1e-3 * sc.extent, count, budget)
            alive = live.sum()
            want += [alive * r[0], alive * r[1], alive * (r[2] + r[3]), alive * r[3], r[4]]
    got = np.array([st.testedNodes, st.visitedNodes, st.evaluatedNodes, st.exactLeaves, st.budgetHits])
    print(f"[budget] counted {got}, walked {want}", flush=True)
    assert np.all(np.abs(got[:4] - want[:4]) <= 0.005 * want[:4] + 0.5)
    assert (got[4] > 0) == (want[4] > 0) and abs(got[4] - want[4]) <= 0.05 * want[4] + 2
    assert st.errorPixels == 0
