"""LBVH builds around the one-workgroup build's limits: sizes around a wave's
128 keys, a power of two and the largest small tree, with many equal codes
(their order is the input's), points and AVPLs, 3D and 6D codes; bit for bit
the oracle's."""
import numpy as np
import pytest

from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import Bvh, DeviceAvpls
from tests.test_gpu_lbvh import build_points, compare

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 63, 64, 65, 127, 128, 129, 255, 257, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097]


def _points(n, seed):
    """Uniform points, a quarter of them copies of a few others."""
    rng = np.random.RandomState(seed)
    p = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    k = rng.rand(n) < 0.25
    p[k] = p[rng.randint(0, min(n, 5), k.sum())]
    return p


@pytest.mark.parametrize("n", SIZES)
def test_points(gpu_ctx, orc, n):
    pos = _points(n, n)
    compare(build_points(gpu_ctx, pos), orc.lbvh_build(pos))


@pytest.mark.parametrize("n", [2, 129, 1025, 4096])
def test_points_with_normals(gpu_ctx, orc, n):
    pos, nrm = _points(n, n), _points(n, n + 1)
    g = build_points(gpu_ctx, pos, nrm, consider_normals=True)
    compare(g, orc.lbvh_build(pos, nrm, consider_normals=True))
    np.testing.assert_array_equal(g["normals"], nrm[g["perm"]])


@pytest.mark.parametrize("n", SIZES)
def test_avpls(gpu_ctx, orc, n):
    sc = S.cornell_256(seed=2, width=8, height=8, num_avpls=n)
    sc.avpl_pos[:] = _points(n, n)
    b = Bvh(gpu_ctx)
    try:
        b.build_avpls(DeviceAvpls.from_scene(sc), seed=n)
        g = b.to_host()
        compare(g, orc.avpl_bvh_build(sc, g["nd_rand"]), node_data=True)
    finally:
        b.close()
