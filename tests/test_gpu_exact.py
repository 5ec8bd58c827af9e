"""The exact gather where its staging and splits can go wrong: images smaller
than a wave and one pixel past a wave's or a block's pixels, AVPL counts
around the 64 that a wave stages and the 32 of the smallest split, no AVPL
with antiradiance and all of them, AVPLs without a direction, pixels without a
normal, lobes whose exponents the power series and powf take.

Against the FP64 kernel on the same inputs.  An FP32 pair carries about 10
roundings (6e-7), of one sign at worst, and a lobe multiplies its cosine's
rounding by its exponent: relative L2 of 1e-5 + 2e-7 * exponent."""
import math

import numpy as np
import pytest

from antiradiancecuts_amd import ffi
from antiradiancecuts_amd import scene as S
from antiradiancecuts_amd.runtime import DeviceAvpls, Gather, default_params, device_array

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


def _check(gpu_ctx, sc, model, tol):
    print(f"[exact] {sc.width}x{sc.height} avpls {sc.num_avpls} model {model}", flush=True)
    g = Gather(gpu_ctx, sc.width, sc.height, sc.materials)
    g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), device_array(sc.albedo4))
    av = DeviceAvpls.from_scene(sc)
    p = default_params(useLightCuts=0, antiradianceMode=0, antiradianceModel=model, coneHalfAngle=math.pi / 18)
    g.run(av, sc.cam, sc.extent, p)
    r64, a64 = g.exact_f64(av, sc.cam, sc.extent, p)
    gpu_ctx.sync()
    rad, anti = (t[:, :3].double().cpu().numpy() for t in (g.radiance, g.antiradiance))
    r64, a64 = r64.cpu().numpy(), a64.cpu().numpy()
    g.close()
    bare = ~sc.nrm4[:, :3].any(1)
    assert _rel(rad[~bare], r64[~bare]) <= tol
    assert _rel(anti[~bare], a64[~bare]) <= tol
    if not sc.materials[:, 6:9].any():
        assert not rad[bare].any() and not anti[bare].any()
    return anti


@pytest.mark.parametrize("model", [ffi.ARC_ANTIRAD_DISK, ffi.ARC_ANTIRAD_CONE])
@pytest.mark.parametrize("w,h,n", [(1, 1, 1), (7, 5, 31), (64, 1, 33), (65, 1, 64), (43, 3, 65), (32, 16, 129),
                                   (27, 19, 1000), (48, 32, 5000)])
@pytest.mark.parametrize("specular", [0, 12])
def test_sizes(gpu_ctx, w, h, n, model, specular):
    sc = S.cornell_256(seed=n, width=w, height=h, num_avpls=n)
    sc.materials[::2, 6:9] = [0.3, 0.25, 0.2] if specular else 0
    sc.materials[::2, 9] = specular
    _check(gpu_ctx, sc, model, 1e-5 + 2e-7 * specular)


@pytest.mark.parametrize("model", [ffi.ARC_ANTIRAD_DISK, ffi.ARC_ANTIRAD_CONE])
@pytest.mark.parametrize("specular", [0, 12])
def test_antiradiance_of_none_and_all(gpu_ctx, model, specular):
    sc = S.cornell_256(seed=1, width=40, height=30, num_avpls=700)
    sc.materials[::2, 6:9] = [0.3, 0.25, 0.2] if specular else 0
    sc.materials[::2, 9] = specular
    sc.avpl_anti[:] = 0
    assert not _check(gpu_ctx, sc, model, 1e-5 + 2e-7 * specular).any()
    sc.avpl_anti[:] = np.random.RandomState(0).uniform(0.1, 1, sc.avpl_anti.shape).astype(np.float32)
    sc.avpl_dir[::5] = 0  # no incident direction: a reflectance of 1, no antiradiance
    sc.nrm4[::7, :3] = 0
    assert _check(gpu_ctx, sc, model, 1e-5 + 2e-7 * specular).any()


@pytest.mark.parametrize("exponent", [0.0, 0.5, 1.0, 7.3, 300.0])
def test_lobes(gpu_ctx, exponent):
    sc = S.cornell_256(seed=9, width=50, height=37, num_avpls=333)
    sc.materials[:, 6:9] = [0.3, 0.25, 0.2]
    sc.materials[:, 9] = exponent
    sc.materials[1, 6:9] = 0
    sc.materials[3, 9] = 40.0
    _check(gpu_ctx, sc, ffi.ARC_ANTIRAD_CONE, 1e-5 + 2e-7 * max(exponent, 40.0))


@pytest.mark.parametrize("model", [ffi.ARC_ANTIRAD_DISK, ffi.ARC_ANTIRAD_CONE])
@pytest.mark.parametrize("exponent", [12.0, 80.0])
def test_antiradiance_of_lobes(gpu_ctx, model, exponent):
    """A pixel's antiradiance is a few AVPLs', all of one sign: each pair's
    relative error is the cosine's rounding (half a unit u = 2^-24) times the
    exponent and 13 u of products (lobe, reflectance, disk or distance,
    antiradiance), and up to 64 of them are added plainly, 20 u for the at most
    20 a pixel has here."""
    sc = S.cornell_256(seed=0, width=64, height=48, num_avpls=500)
    sc.materials[:, 6:9] = [0.3, 0.25, 0.2]
    sc.materials[:, 3:6] = 0
    sc.materials[:, 9] = exponent
    sc.albedo4[:] = 0
    print(f"[exact] antiradiance lobes model {model} exponent {exponent}", flush=True)
    g = Gather(gpu_ctx, sc.width, sc.height, sc.materials)
    g.set_gbuffer(device_array(sc.pos4), device_array(sc.nrm4), device_array(sc.albedo4))
    av = DeviceAvpls.from_scene(sc)
    p = default_params(useLightCuts=0, antiradianceMode=0, antiradianceModel=model, coneHalfAngle=math.pi / 18)
    g.run(av, sc.cam, sc.extent, p)
    _, a64 = g.exact_f64(av, sc.cam, sc.extent, p)
    gpu_ctx.sync()
    anti, a64 = g.antiradiance[:, :3].double().cpu().numpy(), a64.cpu().numpy()
    g.close()
    lit = a64 > 1e-20 * a64.max()
    assert lit.any()
    e = np.abs(anti[lit] / a64[lit] - 1).max() * 2.0 ** 24
    print(f"[exact] largest error {e:.1f} u", flush=True)
    assert e <= 0.5 * exponent + 13 + 20
