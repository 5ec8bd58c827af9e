"""The moment cut's pool memory: its host rules, on the CPU over a counted
device, and on the GPU the case that they are there for."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from antiradiancecuts_amd import ffi
from antiradiancecuts_amd import scene as S

ROOT = Path(__file__).resolve().parent.parent


def test_pool_rules(tmp_path):
    exe = tmp_path / "pool_test"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", f"-I{ROOT / 'antiradiancecuts_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpp" / "pool_test.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0, out.stdout


@pytest.mark.gpu
def test_eager_frames_leave_a_captured_pool(gpu_ctx):
    """A captured view's pool stays where the graph has it while eager frames
    of the same gather ask for several times its chunks and a solid-angle frame
    takes the record buffer: the replays equal the eager frame, and memory
    allocated meanwhile keeps its contents."""
    import torch

    from antiradiancecuts_amd.runtime import Batch, DeviceAvpls, Gather, default_params, device_array

    def params(**kw):
        return default_params(useLightCuts=1, cutMode=ffi.ARC_CUT_ERROR_BOUND, cutPerTile=1,
                              cutEstimator=ffi.ARC_ESTIMATOR_MOMENTS, cutCriterion=ffi.ARC_CRITERION_BOUND,
                              cutImageFloor=0.0, antiradianceModel=ffi.ARC_ANTIRAD_CONE, **kw)

    sc = S.clutter_1080p(seed=41, width=200, height=120, num_avpls=60_000, num_tris=4000)
    b = Batch(gpu_ctx, lanes=1)
    lane = b.lane(0)
    g = Gather(lane, 200, 120, sc.materials)
    try:
        g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), device_array(sc.albedo4))
        av = DeviceAvpls.from_scene(sc)
        loose, tight = params(errorBound=0.05), params(errorBound=2e-4, cutExactCount=0, cutBudget=1 << 20)
        g.run(av, sc.cam, sc.extent, loose)
        lane.sync()
        ref = g.radiance.clone()
        b.capture([(g, av, sc.cam, sc.extent, loose)])
        fills = []
        for rep in range(3):
            for p in (tight, tight, default_params()):
                g.run(av, sc.cam, sc.extent, p)
                lane.sync()
                print(f"[pool] eager frame between replays, rep {rep}", flush=True)
            fills.append(torch.full((16 << 20,), 7.0, device="cuda"))
            g.radiance.fill_(-1.0)
            b.launch()
            gpu_ctx.sync()
            d = (g.radiance[:, :3] - ref[:, :3]).double()
            e = float(d.norm() / ref[:, :3].double().norm())
            print(f"[pool] replay {rep}: rel-L2 {e:.2e}", flush=True)
            # the same cut's sums in the same order
            assert e <= 1e-6
            assert all(bool((f == 7.0).all()) for f in fills)
        assert np.isfinite(g.radiance.cpu().numpy()).all()
    finally:
        g.close()
        b.close()
