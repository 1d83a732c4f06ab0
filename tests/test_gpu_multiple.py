"""Multiple scattering (multiple_scattering.comp:9-93) where its kernel takes
different paths, on the GPU's own density against the FP64 oracle's pass
(precision mode): rows of outer nu texels only (2 slices) and of one inner
slice, wavefronts that straddle slices, and several texels per thread with
outer and inner texels in the same block.

Tolerance 1e-4 (floor 1e-6 x the maximum), the bar of the
pass-by-pass comparisons: a sum of 51 terms read at coordinates rounded at
1e-6 of a texel.
"""
import numpy as np
import pytest

from fuzzyblue_amd import Atmosphere, Builder, Parameters, abi
from oracle import Oracle

pytestmark = pytest.mark.gpu

# (scattering r, mu, mu_s, nu), threads per block (0: default)
CASES = {
    "nu2": ((5, 16, 40, 2), 0),
    "nu3": ((5, 16, 33, 3), 0),
    "straddle": ((4, 16, 65, 5), 0),
    "two_per_thread": ((4, 16, 33, 7), 128),
    "four_per_thread": ((4, 16, 64, 16), 256),
}


@pytest.mark.parametrize("name", CASES)
def test_multiple_paths_vs_oracle(name):
    (r, mu, mus, nu), threads = CASES[name]
    p = Parameters().replace(scattering_r_size=r, scattering_mu_size=mu,
                             scattering_mu_s_size=mus, scattering_nu_size=nu, order=2,
                             flags=abi.FB_FLAG_PRECISE)
    b = Builder(0)
    if threads:
        b.set_tuning(p, multiple_scattering_threads=threads)
    print(f"\n[multiple] {name} {p.scattering_extent()}", flush=True)
    pa = Atmosphere.build(b, None, p)
    pa.wait()
    got = pa.download_scratch("delta_multiple_scattering").reshape(-1, 4)
    J = pa.download_scratch("scattering_density")
    T = pa.atmosphere().download("transmittance")
    pa.close()
    b.close()
    want, _ = Oracle("f64").pass_multiple(p, T, J, np.zeros_like(J))
    want = np.asarray(want, np.float64).reshape(-1, 4)[:, :3]
    x = got[:, :3].astype(np.float64)
    err = np.abs(x - want) / np.maximum(np.abs(want), 1e-6 * np.abs(want).max())
    print(f"  max {err.max():.2e}", flush=True)
    assert err.max() < 1e-4
