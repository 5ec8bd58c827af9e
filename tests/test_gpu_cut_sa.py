"""The solid-angle cut where a wave's shared walk can go wrong: images that do
not fill a tile, trees of two leaves and more, stacks so low that some pixels
of a tile overflow and others do not, flat scenes (every box in the pixels'
plane, decisions at exactly zero), thresholds at both ends, specular
materials.  Counts equal the oracle's traversal pixel by pixel in FP32; the
sums are FP32 sums of at most a few thousand terms of one sign, 1e-4 relative."""
import math

import numpy as np
import pytest

from antiradiancecuts_amd import ffi
from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import DeviceAvpls, Gather, default_params, device_array
from tests.test_oracle_gather import floor_scene

pytestmark = pytest.mark.gpu


def _run(gpu_ctx, sc, thresh, stack):
    print(f"[cut] {sc.width}x{sc.height} avpls {sc.num_avpls} thresh {thresh} stack {stack}", flush=True)
    g = Gather(gpu_ctx, sc.width, sc.height, sc.materials)
    albedo = None if sc.albedo4 is None else device_array(sc.albedo4)
    g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), albedo)
    p = default_params(useLightCuts=1, clusterRefinementThreshold=thresh, stackSize=stack)
    st = g.run(DeviceAvpls.from_scene(sc), sc.cam, sc.extent, p, ffi.ARC_RUN_COUNTERS)
    gpu_ctx.sync()
    tree = g.bvh_to_host()
    rad = g.radiance[:, :3].double().cpu().numpy()
    g.close()
    return st, tree, rad


def _check(gpu_ctx, orc, sc, thresh):
    st, tree, rad = _run(gpu_ctx, sc, thresh, 32)
    orad, oerr, ovis, oev = orc.gather_cut_solid_angle(orc.SceneRef(sc, 0.05), tree, thresh, 32)
    assert (st.visitedNodes, st.evaluatedNodes, st.errorPixels) == (ovis, oev, int(oerr.sum()))
    ok = oerr == 0
    np.testing.assert_allclose(rad[ok], orad[ok], rtol=1e-4, atol=1e-6 * max(np.abs(orad[ok]).max(initial=0.0), 1e-30))
    np.testing.assert_array_equal(rad[~ok], np.tile([1e5, 0, 1e5], ((~ok).sum(), 1)))


def _walk(sc, tree, thresh, size):
    """kernel_bvh's traversal with a stack of `size` entries: nodes visited and evaluated, pixels that overflow."""
    f = np.float32
    with np.errstate(all="ignore"):
        nodes = tree["nodes"]
        lo, hi, rep = nodes["bbMin"].reshape(-1, 3), nodes["bbMax"].reshape(-1, 3), tree["nd_pos"].reshape(-1, 3)
        n = len(lo) + 1
        p, nr = sc.pos4[:, None, :3], sc.nrm4[:, None, :3]
        vis = np.zeros((sc.npix, n - 1), bool)
        for corner in (hi, lo):
            a = corner[None] - p
            inv = f(1) / np.sqrt(a[..., 0] * a[..., 0] + a[..., 1] * a[..., 1] + a[..., 2] * a[..., 2])
            vis |= nr[..., 0] * (a[..., 0] * inv) + nr[..., 1] * (a[..., 1] * inv) + nr[..., 2] * (a[..., 2] * inv) > 0
        e, d = hi - lo, rep[None, n:] - p
        r = f(0.5) * np.sqrt(e[:, 0] * e[:, 0] + e[:, 1] * e[:, 1] + e[:, 2] * e[:, 2])
        dist = np.sqrt(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2])
        below = f(2 * f(3.14159265)) * (f(1) - dist / np.sqrt(r * r + dist * dist)) < f(thresh)
    left, right = nodes["left"].tolist(), nodes["right"].tolist()
    visited = evaluated = 0
    err = np.zeros(sc.npix, bool)
    for q in range(sc.npix):
        v, b, stack = vis[q].tolist(), below[q].tolist(), [-1]
        while stack:
            k = stack.pop()
            if k >= 0:
                evaluated += 1
                continue
            k = -(k + 1)
            visited += 1
            if not v[k]:
                continue
            if b[k]:
                evaluated += 1
                continue
            stack += [left[k], right[k]]
            if len(stack) >= size:
                err[q] = True
                break
    return visited, evaluated, err


@pytest.mark.parametrize("w,h,n,thresh", [
    (1, 1, 2, math.pi / 10), (9, 7, 3, math.pi / 10), (33, 21, 65, 0.05), (70, 50, 3001, math.pi / 10),
    (40, 40, 500, 2 * math.pi + 1e-3), (40, 40, 500, 0.0), (40, 40, 500, 1e-6), (40, 40, 500, 6.28),
])
@pytest.mark.parametrize("specular", [False, True])
def test_ragged_and_extreme(gpu_ctx, orc, w, h, n, thresh, specular):
    sc = S.cornell_256(seed=n, width=w, height=h, num_avpls=n)
    if specular:
        sc.materials[::2, 6:9] = [0.3, 0.25, 0.2]
        sc.materials[::2, 9] = 12.0
    _check(gpu_ctx, orc, sc, thresh)


@pytest.mark.parametrize("stack", [2, 3, 5, 7, 8, 9])
def test_overflow_of_some_pixels(gpu_ctx, stack):
    sc = S.cornell_256(seed=4, width=45, height=30, num_avpls=900)
    st, tree, rad = _run(gpu_ctx, sc, 0.05, stack)
    visited, evaluated, err = _walk(sc, tree, 0.05, stack)
    assert (st.visitedNodes, st.evaluatedNodes, st.errorPixels) == (visited, evaluated, int(err.sum()))
    np.testing.assert_array_equal((rad == [1e5, 0, 1e5]).all(1), err)


def test_boxes_in_the_pixels_plane(gpu_ctx, orc):
    sc = floor_scene(400, 3, W=40, H=30)
    # half of the AVPLs in the pixels' plane, the pixels exactly in it
    flat = np.arange(sc.num_avpls) % 2 == 0
    sc.avpl_pos[flat, 1] = sc.pos4[0, 1]
    _check(gpu_ctx, orc, sc, math.pi / 10)
    sc.avpl_pos[:, 1] = sc.pos4[0, 1]
    _check(gpu_ctx, orc, sc, math.pi / 10)
