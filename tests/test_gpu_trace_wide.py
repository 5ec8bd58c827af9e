"""The eight-wide traversal and the path kernel at the sizes where they can
go wrong: trees of one leaf, of one partly filled node, of exactly eight
children and one more; equal triangles (the lower index wins); rays along
axes and from outside; images that do not fill the last block of pixels; and
path counts around a wave's eight rays, where few paths are traced by the
whole wave and many by eight lanes each.

A hit is the oracle's loop over all triangles: same triangle, same FP32
distance.  A path's AVPLs depend on its number and the seed alone, so those
of the first n of many paths are, bit for bit, those of n paths."""
import ctypes as C
import types

import numpy as np
import pytest

from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import TraceScene, avpls_to_host

pytestmark = pytest.mark.gpu


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _soup(n, seed, flat):
    """n triangles of edge 0.3 around the unit cube; every third one repeats the one before it."""
    rng = np.random.RandomState(seed)
    p0 = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    e = rng.uniform(-0.3, 0.3, (2, n, 3)).astype(np.float32)
    if flat:  # boxes without thickness
        e[:, :, 1] = 0
    p1, p2 = p0 + e[0], p0 + e[1]
    for a in (p0, p1, p2):
        a[2::3] = a[1::3][: len(a[2::3])]
    ts = S.triangle_scene(S.desc(3, 8, 8, 0, 1, 3, 0.0, 1.0, False, 0.3, True, 0, 1e-4, 1e-2))
    m = np.zeros(n, np.int32)
    dark = [k for k, x in enumerate(ts.materials) if not x[:3].any()]
    m[:] = dark[0]
    return types.SimpleNamespace(p0=p0, p1=p1, p2=p2, material=m, materials=ts.materials, light=ts.light)


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 16, 65, 700])
def test_closest_hit_of_small_trees(gpu_ctx, orc, n, flat):
    ts = _soup(n, n, flat)
    rng = np.random.RandomState(100 + n)
    # towards points of random triangles, from inside and far outside, from both sides
    k = rng.randint(0, n, 803)
    w = rng.dirichlet((1, 1, 1), 803).astype(np.float32)
    aim = w[:, :1] * ts.p0[k] + w[:, 1:2] * ts.p1[k] + w[:, 2:] * ts.p2[k]
    org = rng.uniform(-1, 2, (803, 3)).astype(np.float32)
    org[::5] *= 10
    d = aim - org
    d[::3] = np.eye(3, dtype=np.float32)[rng.randint(0, 3, len(d[::3]))] * rng.choice([-1, 1], (len(d[::3]), 1))
    org[::3] = aim[::3] - d[::3] * np.float32(0.75)
    dirs = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    sc = TraceScene(gpu_ctx, ts)
    t, tri = sc.intersect(org, dirs)
    gpu_ctx.sync()
    t, tri = t.cpu().numpy(), tri.cpu().numpy()
    emis, one = np.zeros(256, np.int32), np.zeros(1, np.float32)
    want = np.zeros(803, np.int32)
    dist = np.zeros(803, np.float32)
    for i in range(803):
        want[i] = orc.lib().orc_trace_closest(n, _p(ts.p0), _p(ts.p1), _p(ts.p2), _p(ts.material), _p(emis),
                                              _p(org[i]), _p(dirs[i]), 1e-4, _p(one))
        dist[i] = one[0]
    sc.close()
    assert (want >= 0).any() or n < 3
    np.testing.assert_array_equal(tri, want)
    np.testing.assert_array_equal(t[want >= 0], dist[want >= 0])


def test_paths_do_not_depend_on_their_number(gpu_ctx):
    ts = S.triangle_scene(S.desc(5, 8, 8, 0, 1, 3, 0.0, 1.0, False, 0.3, False, 3000, 1e-3, 1e-2))
    sc = TraceScene(gpu_ctx, ts)
    many = avpls_to_host(sc.shoot(40000, 77), gpu_ctx)  # more than one path per group of lanes
    for n in (1, 3, 7, 8, 9, 31, 33, 1000, 32769):
        few = avpls_to_host(sc.shoot(n, 77), gpu_ctx)
        k = len(few["bounce"])
        assert k == 0 or few["bounce"][0] == 1
        assert len(many["bounce"]) >= k and (len(many["bounce"]) == k or many["bounce"][k] == 1)
        for name in few:
            np.testing.assert_array_equal(few[name], many[name][:k], err_msg=f"{n} paths: {name}")
    sc.close()


@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (5, 1), (37, 21)])
def test_ragged_images(gpu_ctx, w, h):
    """The pixels of a ragged image are those rays that intersect() traces one by one."""
    ts = S.triangle_scene(S.desc(2, 8, 8, 0, 1, 3, 0.0, 1.0, False, 0.3, False, 500, 1e-3, 1e-2), light_quad=False)
    sc = TraceScene(gpu_ctx, ts)
    pos4, nrm4 = sc.gbuffer((0.5, 0.5, 0.02), (0, 0, 1), (0, 1, 0), 0.9, w, h)
    gpu_ctx.sync()
    pos4, nrm4 = pos4.cpu().numpy(), nrm4.cpu().numpy()
    assert np.isfinite(pos4).all() and pos4.shape == (w * h, 4)
    d = pos4[:, :3] - np.float32([0.5, 0.5, 0.02])
    dist = np.linalg.norm(d, axis=1)
    assert (dist > 0).all()  # a closed room: every pixel sees a surface
    t, tri = sc.intersect(np.tile(np.float32([0.5, 0.5, 0.02]), (w * h, 1)), (d / dist[:, None]).astype(np.float32))
    gpu_ctx.sync()
    t = t.cpu().numpy()
    sc.close()
    # the same surface at the same distance: the direction was rounded once (6e-8 of a length of at most 2), and a
    # ray at 1 degree to its surface turns that into 60 times as much
    near = np.abs(t - dist) < 1e-5
    assert near.mean() >= 0.98, near.mean()  # edge pixels may see the other side of an edge
    assert near.all() or w * h > 5
