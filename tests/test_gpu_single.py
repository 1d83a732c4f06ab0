"""Single scattering (single_scattering.comp:9-60) where its kernel takes
different paths, on the GPU's own transmittance against the FP64 oracle's pass
(precision mode): one, two and four texels per thread with rows that fill no
block evenly, transmittance rows of up to two columns per thread (loaded ahead)
and wider ones, and a row too narrow for staging.

FP32 mode, whose quotients by the sample tables' denominators are Markstein's,
against the FP32 restatement on the same cases.

Tolerance 1e-4 (floor 1e-6 x the maximum), the bar of the
pass-by-pass comparisons.
"""
import numpy as np
import pytest

from fuzzyblue_amd import Atmosphere, Builder, Parameters, abi
from oracle import Oracle

pytestmark = pytest.mark.gpu

# (scattering r, mu, mu_s, nu), transmittance mu, threads per block
CASES = {
    "one_texel": ((3, 8, 16, 4), 96, 64),
    "two_texels_three_columns": ((3, 8, 60, 2), 150, 64),
    "four_texels_six_columns": ((3, 8, 33, 7), 346, 64),
    "four_texels_two_columns": ((3, 8, 100, 4), 256, 128),
    "unstaged": ((3, 8, 16, 4), 97, 64),
}


@pytest.mark.parametrize("name", CASES)
def test_single_paths_vs_oracle(name):
    (r, mu, mus, nu), tmu, threads = CASES[name]
    p = Parameters().replace(scattering_r_size=r, scattering_mu_size=mu,
                             scattering_mu_s_size=mus, scattering_nu_size=nu,
                             transmittance_mu_size=tmu, transmittance_r_size=17, order=1,
                             flags=abi.FB_FLAG_PRECISE)
    b = Builder(0)
    b.set_tuning(p, single_scattering_threads=threads)
    print(f"\n[single] {name} {p.scattering_extent()}", flush=True)
    pa = Atmosphere.build(b, None, p)
    pa.wait()
    got = [pa.download_scratch("delta_rayleigh"), pa.download_scratch("delta_mie"),
           pa.atmosphere().download("scattering")]
    T = pa.atmosphere().download("transmittance")
    pa.close()
    b.close()
    for g, want in zip(got, Oracle("f64").pass_single_scattering(p, T)):
        want = np.asarray(want, np.float64).reshape(-1, 4)[:, :3]
        x = g.reshape(-1, 4)[:, :3].astype(np.float64)
        err = np.abs(x - want) / np.maximum(np.abs(want), 1e-6 * np.abs(want).max())
        print(f"  max {err.max():.2e}", flush=True)
        assert err.max() < 1e-4


# Both sides evaluate the same binary32 operations, so what remains is the
# order of the 51 samples' sums and the transmittance taps' interpolation: up
# to 51 roundings of 2^-24, 3e-6.
@pytest.mark.parametrize("name", CASES)
def test_single_paths_vs_restatement(name):
    (r, mu, mus, nu), tmu, threads = CASES[name]
    p = Parameters().replace(scattering_r_size=r, scattering_mu_size=mu,
                             scattering_mu_s_size=mus, scattering_nu_size=nu,
                             transmittance_mu_size=tmu, transmittance_r_size=17, order=1)
    b = Builder(0)
    b.set_tuning(p, single_scattering_threads=threads)
    print(f"\n[single] fp32 {name} {p.scattering_extent()}", flush=True)
    pa = Atmosphere.build(b, None, p)
    pa.wait()
    got = [pa.download_scratch("delta_rayleigh"), pa.download_scratch("delta_mie"),
           pa.atmosphere().download("scattering")]
    T = pa.atmosphere().download("transmittance")
    pa.close()
    b.close()
    for g, want in zip(got, Oracle("f32").pass_single_scattering(p, T)):
        want = np.asarray(want, np.float64).reshape(-1, 4)[:, :3]
        x = g.reshape(-1, 4)[:, :3].astype(np.float64)
        err = np.abs(x - want) / np.maximum(np.abs(want), 1e-6 * np.abs(want).max())
        print(f"  max {err.max():.2e}", flush=True)
        assert err.max() < 3e-6
