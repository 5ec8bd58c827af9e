"""The key sort at its tiles' edges (2048 keys, waves of 256): sizes around
multiples of both, keys all equal, of two digits, and random; the order of
equal keys is the input's.  Through the builds that use it (more than 4096
points): codes and permutation equal numpy's stable sort of the codes."""
import numpy as np
import pytest

from antiradiancecuts_amd.runtime import Bvh, device_array

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["random", "equal", "two"])
@pytest.mark.parametrize("n", [4097, 4351, 4352, 4353, 6143, 6144, 6145, 8191, 8192, 8193, 100_003])
def test_sorted_and_stable(gpu_ctx, orc, n, kind):
    rng = np.random.RandomState(n)
    p = rng.rand(n, 3).astype(np.float32)
    if kind == "equal":
        p[:] = p[0]
    elif kind == "two":
        p[:] = p[rng.randint(0, 2, n)]
    b = Bvh(gpu_ctx)
    try:
        b.build_points(device_array(p))
        g = b.to_host()
    finally:
        b.close()
    code = np.empty(n, np.uint32)
    code[g["perm"]] = g["codes"]  # the input's codes, if perm is a permutation
    assert np.array_equal(np.sort(g["perm"]), np.arange(n))
    order = np.argsort(code, kind="stable")
    np.testing.assert_array_equal(g["perm"], order)
    np.testing.assert_array_equal(g["codes"], code[order])
    np.testing.assert_array_equal(g["codes"], orc.lbvh_build(p)["codes"])


@pytest.mark.parametrize("kind", ["random", "two"])
@pytest.mark.parametrize("n", [129_025, 131_071, 131_072, 131_073, 133_121, 1_048_576, 1_048_577, 2_097_153])
def test_tile_counts(gpu_ctx, n, kind):
    """At 64 tiles, the most whose counts the scatter sums itself, and at 512
    and 1024, a block's width of the scan once and twice."""
    rng = np.random.RandomState(n)
    p = rng.rand(n, 3).astype(np.float32)
    if kind == "two":
        p[:] = p[rng.randint(0, 2, n)]
    b = Bvh(gpu_ctx)
    try:
        b.build_points(device_array(p))
        g = b.to_host()
    finally:
        b.close()
    assert np.array_equal(np.bincount(g["perm"], minlength=n), np.ones(n, np.int64))
    code = np.empty(n, np.uint32)
    code[g["perm"]] = g["codes"]
    np.testing.assert_array_equal(g["perm"], np.argsort(code, kind="stable"))
    assert np.all(np.diff(g["codes"].astype(np.int64)) >= 0)
