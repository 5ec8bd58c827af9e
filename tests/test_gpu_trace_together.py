"""Many rays over trees of few nodes: a wave's 64 rays go through the tree
together.  What they find is, bit for bit, what a ray finds in its eight lanes:
the same rays in a call of fewer, the same picture of a scene whose tree is
larger because of triangles that no ray reaches, the first paths of a shoot of
fewer."""
import types

import numpy as np
import pytest

from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import TraceScene, avpls_to_host

pytestmark = pytest.mark.gpu


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
    ts = _room(True)
    dark = [k for k, x in enumerate(ts.materials) if not x[:3].any()]
    return types.SimpleNamespace(p0=p0, p1=p1, p2=p2, material=np.full(n, dark[0], np.int32), materials=ts.materials,
                                 light=ts.light)


def _room(boxes=False, clutter=0):
    return S.triangle_scene(S.desc(5, 8, 8, 0, 1, 3, 0.0, 1.0, False, 0.3, boxes, clutter, 1e-3, 1e-2))


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 16])
def test_rays(gpu_ctx, n, flat):
    ts = _soup(n, n, flat)
    rng = np.random.RandomState(200 + n)
    k = rng.randint(0, n, 801)
    w = rng.dirichlet((1, 1, 1), 801).astype(np.float32)
    aim = w[:, :1] * ts.p0[k] + w[:, 1:2] * ts.p1[k] + w[:, 2:] * ts.p2[k]
    org = rng.uniform(-1, 2, (801, 3)).astype(np.float32)
    d = aim - org
    d[::3] = np.eye(3, dtype=np.float32)[rng.randint(0, 3, len(d[::3]))] * rng.choice([-1, 1], (len(d[::3]), 1))
    org[::3] = aim[::3] - d[::3] * np.float32(0.75)
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    sc = TraceScene(gpu_ctx, ts)
    t0, tri0 = (x.cpu().numpy() for x in sc.intersect(org, d))
    for m in (200000, 200001, 200063):
        order = rng.randint(0, 801, m)
        t, tri = (x.cpu().numpy() for x in sc.intersect(org[order], d[order]))
        np.testing.assert_array_equal(tri, tri0[order])
        np.testing.assert_array_equal(t.view(np.int32), t0[order].view(np.int32))
    sc.close()


@pytest.mark.parametrize("boxes,clutter", [(False, 0), (True, 0), (False, 200)])
@pytest.mark.parametrize("w,h", [(613, 331), (200000, 1), (3, 66667)])
def test_pictures(gpu_ctx, boxes, clutter, w, h):
    ts = _room(boxes, clutter)
    far = np.random.RandomState(1).uniform(3, 4, (4000, 3)).astype(np.float32)  # outside the closed room
    add = lambda a, dx: np.concatenate([a, far + np.float32(dx)])  # noqa: E731
    big = types.SimpleNamespace(
        p0=add(ts.p0, (0, 0, 0)), p1=add(ts.p1, (0.01, 0, 0)), p2=add(ts.p2, (0, 0.01, 0)),
        material=np.concatenate([ts.material, np.full(4000, ts.material[0], ts.material.dtype)]),
        materials=ts.materials, light=ts.light)
    got = []
    for scene in (ts, big):
        sc = TraceScene(gpu_ctx, scene)
        pos4, nrm4 = sc.gbuffer((0.5, 0.5, 0.02), (0.2, -0.1, 1), (0, 1, 0), 0.9, w, h)
        got.append((pos4.cpu().numpy(), nrm4.cpu().numpy()))
        sc.close()
    assert (got[0][0][:, :3] != got[0][0][0, :3]).any()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a.view(np.int32), b.view(np.int32))


@pytest.mark.parametrize("boxes,clutter", [(False, 0), (True, 0), (False, 50)])
def test_paths(gpu_ctx, boxes, clutter):
    sc = TraceScene(gpu_ctx, _room(boxes, clutter))
    few = avpls_to_host(sc.shoot(90001, 77), gpu_ctx)
    k = len(few["bounce"])
    assert k > 90001
    for n in (110001, 300000):
        many = avpls_to_host(sc.shoot(n, 77), gpu_ctx)
        assert many["bounce"][k] == 1
        for name in few:
            np.testing.assert_array_equal(many[name][:k], few[name], err_msg=f"{n} paths: {name}")
    sc.close()
