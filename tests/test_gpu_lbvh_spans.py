"""The refit's climb across blocks and spans: leaf counts around a block (1024
leaves), spans of 8 and 64 blocks, points whose codes are all equal (the tree
splits by index alone), half equal, or share long prefixes at a boundary;
AvplBvh node data bit for bit the oracle's.  (The light cut's records climb
through the same kernels; their sums are in the images that the cut's tests
compare.)"""
import numpy as np
import pytest

from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import Bvh, DeviceAvpls
from tests.test_gpu_lbvh import compare

pytestmark = pytest.mark.gpu


def _points(n, kind):
    rng = np.random.RandomState(n)
    p = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    if kind == "equal":
        p[:] = p[0]
    elif kind == "half":
        p[n // 3:] = p[0]
    elif kind == "clustered":  # codes that differ in the last bits only, and a few far ones
        p *= 1e-3
        p[::97] = rng.uniform(-1, 1, (len(p[::97]), 3))
    return p


@pytest.mark.parametrize("kind", ["uniform", "equal", "half", "clustered"])
@pytest.mark.parametrize("n", [1024, 1025, 2049, 8191, 8192, 8193, 9217, 20000, 65536, 65537, 70000])
def test_avpl_tree(gpu_ctx, orc, n, kind):
    print(f"[lbvh] {kind} {n}", flush=True)
    sc = S.cornell_256(seed=2, width=8, height=8, num_avpls=n)
    sc.avpl_pos[:] = _points(n, kind)
    b = Bvh(gpu_ctx)
    try:
        b.build_avpls(DeviceAvpls.from_scene(sc), seed=n)
        g = b.to_host()
        b.check_integrity()
    finally:
        b.close()
    compare(g, orc.avpl_bvh_build(sc, g["nd_rand"]), node_data=True)
