"""The moment cut's serial path: tiles that find the pool full, tiles that meet
their budget, small budgets, and the order of the tiles by the last cut's costs.

Two ways to one cut sum the same FP32 terms in other orders: relative L2 of
1e-5.  A decision whose bound lies on its threshold may turn, about one in 1e6,
and moves the counts by a subtree: 0.5 %.
"""
import numpy as np
import pytest

from antiradiancecuts_amd import ffi
from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import Batch, DeviceAvpls, Gather, default_params, device_array

pytestmark = pytest.mark.gpu


def params(**kw):
    base = dict(useLightCuts=1, cutMode=ffi.ARC_CUT_ERROR_BOUND, cutPerTile=1, cutEstimator=ffi.ARC_ESTIMATOR_MOMENTS,
                cutCriterion=ffi.ARC_CRITERION_BOUND, cutImageFloor=0.0, antiradianceModel=ffi.ARC_ANTIRAD_CONE)
    base.update(kw)
    return default_params(**base)


def rig(ctx, w, h, n, seed=13):
    sc = S.clutter_1080p(seed=seed, width=w, height=h, num_avpls=n, num_tris=4000)
    g = Gather(ctx, w, h, sc.materials)
    g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), device_array(sc.albedo4))
    return sc, g, DeviceAvpls.from_scene(sc)


def frame(ctx, sc, g, av, p):
    st = g.run(av, sc.cam, sc.extent, p, ffi.ARC_RUN_COUNTERS)
    ctx.sync()
    assert st.errorPixels == 0
    counts = np.array([st.testedNodes, st.visitedNodes, st.evaluatedNodes, st.exactLeaves], np.float64)
    return g.radiance[:, :3].cpu().numpy(), counts, st.budgetHits


def rel(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("w,h,n,count,criterion", [
    (1003, 811, 20_000, 16, ffi.ARC_CRITERION_BOUND),      # ragged tiles
    (1003, 811, 6_000, 128, ffi.ARC_CRITERION_BOUND),      # range chunks of several parts
    (800, 600, 30_000, 0, ffi.ARC_CRITERION_EXPANSION),    # down to single leaves
])
def test_full_pool(gpu_ctx, w, h, n, count, criterion):
    """A pool of one chunk per tile holds 16384; each of the 7500 to 12852 tiles
    asks for eight at once, so most find it full: in the first frame as they
    come, in the next ones all tiles are cut serially."""
    sc, g, av = rig(gpu_ctx, w, h, n)
    try:
        p = params(cutExactCount=count, cutCriterion=criterion)
        frame(gpu_ctx, sc, g, av, p)
        ref, want, _ = frame(gpu_ctx, sc, g, av, p)
        again, _, _ = frame(gpu_ctx, sc, g, av, p)
        assert np.array_equal(ref, again) and np.isfinite(ref).all() and ref.max() > 0
        g.set_estimate_pool(1)
        last = None
        for k in range(4):
            rad, counts, hits = frame(gpu_ctx, sc, g, av, p)
            print(f"[serial] {w}x{h} n={n} frame {k}: rel-L2 {rel(rad, ref):.2e}, counts {counts / want}", flush=True)
            assert hits == 0 and rel(rad, ref) <= 1e-5
            assert np.all(np.abs(counts - want) <= 0.005 * want + 0.5)
            if k > 1:  # all tiles serial, ordered by the costs of different frames
                assert np.array_equal(rad, last)
            last = rad
    finally:
        g.close()


@pytest.mark.parametrize("w,h,n,bound,budget", [
    (203, 117, 20_000, 1e-2, 512),       # a small budget: no pool at all
    (500, 301, 20_000, 1e-3, 9_000),     # most tiles meet it: decided first, then cut serially
    (500, 301, 20_000, 1e-2, 65_536),    # none does
])
def test_frames_repeat(gpu_ctx, w, h, n, bound, budget):
    """The counts hold to the first frame's, also where the tiles that meet
    their budget change kernels after it (the serial cut counts up to 128 kept
    nodes before it drops those that face away), and later frames, whatever the
    order of their tiles, are equal bit for bit."""
    sc, g, av = rig(gpu_ctx, w, h, n)
    try:
        p = params(errorBound=bound, cutBudget=budget)
        images, counts, hits = zip(*[frame(gpu_ctx, sc, g, av, p) for _ in range(4)])
    finally:
        g.close()
    print(f"[serial] {w}x{h} budget {budget}: counts {[(c / counts[0]).round(4).tolist() for c in counts]} hits {hits}",
          flush=True)
    assert (hits[0] > 0) == (budget < 65_536)
    for k in range(1, 4):
        assert np.all(np.abs(counts[k] - counts[0]) <= (0.005 + 128 / budget) * counts[0] + 0.5)
        assert (hits[k] > 0) == (hits[0] > 0)
    assert np.array_equal(images[2], images[3])
    if budget != 9_000:
        assert np.array_equal(images[0], images[2])


@pytest.mark.parametrize("budgets", [(512, 65_536, 65_536), (512, 512, 512), (65_536, 4096, 9_000)])
def test_one_launch_of_uneven_budgets(gpu_ctx, budgets):
    """Views whose tiles are cut serially in one launch with views whose are
    not: each replay gives every view's eager image."""
    shapes = [(203, 117, 20_000), (320, 200, 9_000), (96, 64, 30_000)]
    b = Batch(gpu_ctx, lanes=2)
    views, ref = [], []
    try:
        for k, ((w, h, n), budget) in enumerate(zip(shapes, budgets)):
            p = params(errorBound=1e-3, cutBudget=budget)
            sc, g, av = rig(gpu_ctx, w, h, n, seed=40 + k)
            ref.append(frame(gpu_ctx, sc, g, av, p)[0])
            g.close()
            sc, g, av = rig(b.lane(k), w, h, n, seed=40 + k)  # has run no frame before the capture
            views.append((g, av, sc.cam, sc.extent, p))
        print(f"[serial] one launch, budgets {budgets}", flush=True)
        b.set_one_cut_launch(True)
        b.capture(views)
        for rep in range(3):
            for g, *_ in views:
                g.radiance.fill_(-1.0)
            b.launch()
            gpu_ctx.sync()
            for k, (g, *_rest) in enumerate(views):
                e = rel(g.radiance[:, :3].cpu().numpy(), ref[k])
                print(f"[serial] replay {rep} view {k}: rel-L2 {e:.2e}", flush=True)
                assert e <= 1e-5
    finally:
        for g, *_ in views:
            g.close()
        b.close()
