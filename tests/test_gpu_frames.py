"""Frames whose pixels end inside a thread's group of rays (four pixels a
stride apart), inside a block's first stride and just past a block: the rays
depend on the pixel's index only, so a frame's pixels equal those of a longer
frame bit for bit, and nothing is written past its end.  Cameras on the LUT
slice path and above the atmosphere (per-ray lookups)."""
import numpy as np
import pytest

from fuzzyblue_amd import Atmosphere, DeviceBuffer, Parameters, Renderer, synchronize
from fuzzyblue_amd.params import DUMP_SIZES

pytestmark = pytest.mark.gpu

LONG, GUARD = 9000, 64


@pytest.mark.parametrize("altitude", [2.0, 75.0])
def test_frame_ends(builder, altitude):
    pa = Atmosphere.build(builder, None, Parameters().replace(**DUMP_SIZES))
    pa.wait()
    a = pa.assert_ready()
    r = Renderer(builder)
    alt = DeviceBuffer.from_array(np.array([altitude], np.float32))
    zen = DeviceBuffer.from_array(np.array([1.0], np.float32))

    def frame(pixels):
        out = DeviceBuffer.from_array(np.full((pixels + GUARD, 4), -7.0, np.float32))
        r.frames(None, a, alt, zen, 1, pixels, 5, out)
        synchronize()
        return out.to_array(np.float32, (pixels + GUARD, 4))

    print(f"\n[frames] altitude {altitude}", flush=True)
    want = frame(LONG)
    for pixels in (1, 255, 257, 769, 1023, 1025, 4095, 4097):
        got = frame(pixels)
        assert np.array_equal(got[:pixels], want[:pixels]), pixels
        assert np.all(got[pixels:] == -7.0), pixels
    a.close()
