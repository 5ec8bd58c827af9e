"""The tuner times only the knobs that a kernel's speed depends on."""
import types

from antiradiancecuts_amd import autotune, ffi


class _Gather:
    """Stands for a gather whose frames get faster with every frame, so that any candidate that is timed wins."""

    def __init__(self):
        self.ms, self.shapes, self.pools = 1000.0, [], []

    def set_launch_shape(self, cut_stack, anti_chunk):
        self.shapes.append((cut_stack, anti_chunk))

    def set_estimate_pool(self, chunks):
        self.pools.append(chunks)

    def run(self, avpls, cam, extent, p, flags):
        self.ms -= 1.0
        return types.SimpleNamespace(errorPixels=0, msTotal=self.ms)


def test_no_candidate_names_a_stack():
    p = ffi.arc_gather_params()
    p.useLightCuts, p.cutMode, p.cutEstimator = 1, ffi.ARC_CUT_ERROR_BOUND, ffi.ARC_ESTIMATOR_MOMENTS
    p.antiradianceMode = ffi.ARC_ANTI_CLUSTERED
    g = _Gather()
    best, sched, table = autotune.tune(g, None, None, 0.0, p, reps=2)
    default = autotune.Schedule()
    assert sched.cut_stack == default.cut_stack and {s for s, _ in g.shapes} == {default.cut_stack}
    assert {a for _, a in g.shapes} == {1536, 768, 3072} and set(g.pools) == {0, 32}
    assert not any(name.startswith("cut_stack") for name, _ in table)
    assert (sched.anti_chunk, sched.estimate_pool) == (3072, 32)  # the last ones timed
