"""Scattering density (scattering_density.comp:10-155) where its kernel takes
different paths, in both arithmetic modes, on the GPU's own inputs against
the oracle's pass:

  * nu extents with only outer texels (2), one inner slice (3), and an even
    and an odd number of slices;
  * theta-split sets (under 65,536 texels), and one, two, four, six and
    seven texels per thread, some not filling their wavefronts evenly;
  * an Earth-like planet (most ground rows meet no knot of the irradiance
    LUT) and a small one with a thick atmosphere under a fine irradiance LUT
    (rows of one knot and of many).

FP32 mode leaves out the Earth-like planet at the sizes past the theta-split
limit: at extents that are no powers of two the binary32 texture coordinate
of a lookup at mu_s_min falls a few 1e-5 of a texel into the previous nu
slice, whose last texel is up to 1e7 times brighter there (see
test_gpu_shapes.py), so the restatement itself is off.

Tolerance 1e-4 (floor 1e-6 x the sampled texels' maximum), the bar of the
pass-by-pass comparisons: a sum of 512 terms, each rounded at 1e-7 and read
at coordinates rounded at 1e-6 of a texel.
"""
import numpy as np
import pytest

from fuzzyblue_amd import Atmosphere, Parameters, abi
from oracle import Oracle

pytestmark = pytest.mark.gpu

SIZES = {
    "split_nu2": dict(scattering_r_size=4, scattering_mu_size=16, scattering_mu_s_size=8,
                      scattering_nu_size=2),
    "split_nu3": dict(scattering_r_size=4, scattering_mu_size=32, scattering_mu_s_size=9,
                      scattering_nu_size=3),
    "one_nu5": dict(scattering_r_size=16, scattering_mu_size=64, scattering_mu_s_size=13,
                    scattering_nu_size=5),
    "pair_nu6": dict(scattering_r_size=8, scattering_mu_size=128, scattering_mu_s_size=11,
                     scattering_nu_size=6),
    "four_nu6": dict(scattering_r_size=32, scattering_mu_size=72, scattering_mu_s_size=43,
                     scattering_nu_size=6),
    "six_nu8": dict(scattering_r_size=32, scattering_mu_size=72, scattering_mu_s_size=43,
                    scattering_nu_size=8),
    "seven_nu9": dict(scattering_r_size=32, scattering_mu_size=72, scattering_mu_s_size=43,
                      scattering_nu_size=9),
}
PLANETS = {
    "earth": {},
    "small": dict(bottom_radius=500.0, top_radius=700.0, irradiance_mu_s_size=256),
}


CASES = [(s, p, m) for s in SIZES for p in PLANETS for m in (True, False)
         if m or p == "small" or s.startswith("split")]


@pytest.mark.parametrize("size,planet,precise", CASES,
                         ids=[f"{s}-{p}-{'precise' if m else 'fp32'}" for s, p, m in CASES])
def test_density_paths_vs_oracle(builder, size, planet, precise):
    p = Parameters().replace(**SIZES[size], **PLANETS[planet],
                             flags=abi.FB_FLAG_PRECISE if precise else 0)
    o = Oracle("f64" if precise else "f32")
    w, h, d = p.scattering_extent()
    rng = np.random.default_rng(7)
    idx = np.sort(rng.choice(w * h * d, min(w * h * d, 2048), replace=False))
    print(f"\n[density] {size} {planet} {'precise' if precise else 'fp32'}", flush=True)
    got = {}
    for order in (1, 2, 3):
        pa = Atmosphere.build(builder, None, p.replace(order=order))
        pa.wait()
        got[order] = {k: pa.download_scratch(k) for k in (
            "delta_irradiance", "delta_rayleigh", "delta_mie", "delta_multiple_scattering",
            "scattering_density")}
        T = pa.atmosphere().download("transmittance")
        pa.close()
    for order in (2, 3):
        prev = got[order - 1]
        want = np.asarray(o.density_texels(p, order, T, prev["delta_rayleigh"],
                                           prev["delta_mie"],
                                           prev["delta_multiple_scattering"],
                                           prev["delta_irradiance"], idx), np.float64)[..., :3]
        x = got[order]["scattering_density"].reshape(-1, 4)[idx, :3].astype(np.float64)
        err = np.abs(x - want) / np.maximum(np.abs(want), 1e-6 * np.abs(want).max())
        print(f"  order {order}: max {err.max():.2e}", flush=True)
        assert err.max() < 1e-4


def test_density_error_with_a_sharp_mie_peak(builder):
    """At g = 0.95 an ulp of omega.omega_i near the Mie peak moves a direction's
    weight by 5e-6, so the density's error against 64 bits follows how that
    cosine is rounded: an RMS of 1.10e-6 with the direction table's products,
    1.25e-6 where sin(theta) omega.x is rounded once for a whole theta row.
    The bar lies between."""
    p = Parameters().replace(scattering_r_size=8, scattering_mu_size=64,
                             scattering_mu_s_size=32, scattering_nu_size=8,
                             mie_phase_function_g=0.95, mie_scattering=[0.02] * 3,
                             mie_extinction=[0.022] * 3, flags=abi.FB_FLAG_PRECISE)
    w, h, d = p.scattering_extent()
    idx = np.sort(np.random.default_rng(7).choice(w * h * d, 4096, replace=False))
    got = {}
    for order in (2, 3):
        pa = Atmosphere.build(builder, None, p.replace(order=order))
        pa.wait()
        got[order] = {k: pa.download_scratch(k) for k in (
            "delta_irradiance", "delta_rayleigh", "delta_mie", "delta_multiple_scattering",
            "scattering_density")}
        T = pa.atmosphere().download("transmittance")
        pa.close()
    prev = got[2]
    want = np.asarray(Oracle("f64").density_texels(
        p, 3, T, prev["delta_rayleigh"], prev["delta_mie"], prev["delta_multiple_scattering"],
        prev["delta_irradiance"], idx), np.float64)[..., :3]
    x = got[3]["scattering_density"].reshape(-1, 4)[idx, :3].astype(np.float64)
    err = (x - want) / np.maximum(np.abs(want), 1e-6 * np.abs(want).max())
    rms = np.sqrt((err ** 2).mean())
    print(f"\n[density] g 0.95: RMS {rms:.3e}", flush=True)
    assert rms < 1.18e-6
