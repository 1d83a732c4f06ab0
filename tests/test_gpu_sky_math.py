"""The sky lookups' square root, reciprocal and quotients (sky_math.hpp) against
the compiler's IEEE operations on the device, bit for bit: the root and the
reciprocal at every binary32 value of their ranges, the quotients on pairs of
boundary values, on random pairs and with extreme lanes among ordinary ones.
Exact: no tolerance."""
import ctypes as C

import numpy as np
import pytest

from fuzzyblue_amd import DeviceBuffer
from fuzzyblue_amd.build import CHECKS_LIB

pytestmark = pytest.mark.gpu


def call(fn, *args):
    count, example = C.c_ulonglong(), (C.c_float * 2)()
    f = getattr(C.CDLL(CHECKS_LIB), fn)
    assert f(*args, C.byref(count), example) == 0
    return count.value, [x.hex() for x in example]


def quotients(a, b, kind):
    a, b = (np.ascontiguousarray(x, np.float32) for x in (a, b))
    da, db = DeviceBuffer.from_array(a), DeviceBuffer.from_array(b)
    return call("fbc_quotient", da.ptr, db.ptr, C.c_size_t(a.size), C.c_int(kind))


@pytest.mark.parametrize("fn", ["fbc_sqrt", "fbc_reciprocal"])
def test_every_argument(builder, fn):
    print(f"\n[sky math] {fn}", flush=True)
    count, example = call(fn)
    assert count == 0, example


def boundary_values():
    v = [0.0, 1.0, 1.5, 3.0, np.inf, np.nan, 2.0 ** -149, 2.0 ** -126]
    for e in (-100, -80, -60, 0, 60, 100, 127):
        x = np.float32(2.0 ** e)
        v += [x, np.nextafter(x, np.float32(0)), np.nextafter(x, np.float32(np.inf))]
    v = np.array(v, np.float32)
    return np.concatenate([v, -v])


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_quotients_of_boundary_values(builder, kind):
    v = boundary_values()
    a, b = np.repeat(v, v.size), np.tile(v, v.size)
    # Each pair with a wavefront of its own, then all mixed.
    for x, y in ((np.repeat(a, 64), np.repeat(b, 64)), (a, b)):
        count, example = quotients(x, y, kind)
        assert count == 0, example


def random_values(rng, n, lo, hi):
    x = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(lo, hi, n)
    return (x * np.where(rng.random(n) < 0.5, -1, 1)).astype(np.float32)


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_quotients_of_random_pairs(builder, kind):
    rng = np.random.default_rng(11)
    n = 1 << 22
    for lo, hi in ((-2, 2), (-60, 60), (-80, 46)):
        count, example = quotients(random_values(rng, n, lo, hi), random_values(rng, n, lo, hi),
                                   kind)
        assert count == 0, example


def test_quotients_beside_an_extreme_lane(builder):
    rng = np.random.default_rng(12)
    n = 1 << 20
    a, b = random_values(rng, n, -20, 20), random_values(rng, n, -20, 20)
    a[::64] = random_values(rng, n // 64, -126, -90)
    b[32::128] = np.inf
    for kind in (1, 2):
        count, example = quotients(a, b, kind)
        assert count == 0, example
