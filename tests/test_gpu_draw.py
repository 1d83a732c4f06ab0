"""Draws large enough for the per-draw LUT slice (1500 x 1001 pixels, which
fill no block evenly) against the FP32 restatement of render_sky.frag:24-35,
with and without geometry behind each pixel, the same draw with a sun vector
longer than 1, which the slice does not cover, and draws with no geometry at
all, whose pixels below the horizontal take the far end of an infinite segment
at the bottom (a NaN of the restatement's binary32, clamped).

Tolerances are those of the small draw's comparison (transmittance 1e-4 at a
floor of 1e-6 of the maximum, radiance 1e-3 at 1e-4).  One pixel in a thousand
may exceed them: the horizon, one row of the 1001, is where an ulp of the view
direction moves a lookup between the two halves of the scattering LUT.
"""
import ctypes as C

import numpy as np
import pytest

from fuzzyblue_amd import (Atmosphere, DeviceBuffer, DrawParameters, Parameters, Renderer, abi,
                           synchronize)
from fuzzyblue_amd.params import DUMP_SIZES
from oracle import Oracle

pytestmark = pytest.mark.gpu

W, H = 1500, 1001


def rel_err(x, y, floor):
    x = np.asarray(x, np.float64)[..., :3]
    y = np.asarray(y, np.float64)[..., :3]
    return np.abs(x - y) / np.maximum(np.abs(y), floor * max(np.abs(y).max(), 1e-30))


@pytest.mark.parametrize("sun_length", [1.0, 1.01])
def test_large_draw_matches_fragment_shader(builder, sun_length):
    p = Parameters().replace(**DUMP_SIZES)
    pa = Atmosphere.build(builder, None, p)
    pa.wait()
    a = pa.assert_ready()
    T = a.download("transmittance").astype(np.float64)
    S = a.download("scattering").astype(np.float64)
    # Inverse of a reverse-Z infinite perspective for a camera 2 km up looking
    # along +x (column-major, [column][row]), in metres.
    near = 0.1
    ivp = np.zeros((4, 4), np.float32)
    ivp[0] = [0.0, -0.75, 0.0, 0.0]
    ivp[1] = [0.0, 0.0, -0.5, 0.0]
    ivp[2] = [0.0, 0.0, 6362e3 / near, 1.0 / near]
    ivp[3] = [1.0, 0.0, 0.0, 0.0]
    draw = DrawParameters(inverse_viewproj=ivp.tolist(), camera_position=[0.0, 0.0, 6362.0],
                          sun_direction=[0.6 * sun_length, 0.0, 0.8 * sun_length])
    depth = np.random.default_rng(3).uniform(near / 50e3, near / 500.0, (H, W)).astype(np.float32)
    depth[: H // 2] = 0.0  # upper half: infinitely far
    color, tr = DeviceBuffer(W * H * 16), DeviceBuffer(W * H * 16)
    print(f"\n[draw] {W}x{H} sun {sun_length}", flush=True)
    Renderer(builder).draw(None, a, draw, W, H, color, tr, depth=DeviceBuffer.from_array(depth))
    synchronize()
    g_c = color.to_array(np.float32, (H, W, 4))
    g_t = tr.to_array(np.float32, (H, W, 4))
    a.close()
    o_c, o_t = Oracle("f32").render_frame(p, T, S, ivp, draw.camera_position,
                                           draw.sun_direction, W, H, depth=depth)
    t_bad = (rel_err(g_t, o_t, 1e-6) > 1e-4).any(-1).mean()
    c_bad = (rel_err(g_c, o_c, 1e-4) > 1e-3).any(-1).mean()
    print(f"  pixels outside: transmittance {t_bad:.2e}, radiance {c_bad:.2e}", flush=True)
    assert t_bad < 1e-3 and c_bad < 1e-3
    assert np.all(g_c[..., 3] == 0.0) and np.all(g_t[..., 3] == 1.0)


def view_along_x(near=0.1):
    """Inverse of a reverse-Z infinite perspective for a camera 2 km up looking
    along +x (column-major, [column][row]), in metres."""
    ivp = np.zeros((4, 4), np.float32)
    ivp[0] = [0.0, -0.75, 0.0, 0.0]
    ivp[1] = [0.0, 0.0, -0.5, 0.0]
    ivp[2] = [0.0, 0.0, 6362e3 / near, 1.0 / near]
    ivp[3] = [1.0, 0.0, 0.0, 0.0]
    return ivp


# (Even extents: on a centre line the far point at depth 0 is 0/0.)
@pytest.mark.parametrize("size", [(1500, 1000), (150, 100)], ids=["slice", "direct"])
def test_draw_without_geometry_matches_fragment_shader(builder, size):
    w, h = size
    p = Parameters().replace(**DUMP_SIZES)
    pa = Atmosphere.build(builder, None, p)
    pa.wait()
    a = pa.assert_ready()
    T = a.download("transmittance").astype(np.float64)
    S = a.download("scattering").astype(np.float64)
    ivp = view_along_x()
    draw = DrawParameters(inverse_viewproj=ivp.tolist(), camera_position=[0.0, 0.0, 6362.0],
                          sun_direction=[0.6, 0.0, 0.8])
    color, tr = DeviceBuffer(w * h * 16), DeviceBuffer(w * h * 16)
    print(f"\n[draw] {w}x{h} without depth", flush=True)
    Renderer(builder).draw(None, a, draw, w, h, color, tr)
    synchronize()
    g_c = color.to_array(np.float32, (h, w, 4))
    g_t = tr.to_array(np.float32, (h, w, 4))
    a.close()
    o_c, o_t = Oracle("f32").render_frame(p, T, S, ivp, draw.camera_position,
                                           draw.sun_direction, w, h)
    t_bad = (rel_err(g_t, o_t, 1e-6) > 1e-4).any(-1)
    c_bad = (rel_err(g_c, o_c, 1e-4) > 1e-3).any(-1)
    limit = max(1e-3, 1.0 / h)  # the horizon's row (see above)
    print(f"  pixels outside: transmittance {t_bad.mean():.2e}, radiance {c_bad.mean():.2e}",
          flush=True)
    assert np.isfinite(g_c).all() and np.isfinite(g_t).all()
    assert t_bad.mean() <= limit and c_bad.mean() <= limit


def test_large_draw_on_the_legacy_stream_beside_a_captured_one(builder):
    """While a blocking stream is captured the legacy stream has no capture
    status and must not allocate: a large draw there goes without the slice."""
    w, h = 1500, 1000
    pa = Atmosphere.build(builder, None, Parameters().replace(**DUMP_SIZES))
    pa.wait()
    a = pa.assert_ready()
    paths = {line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line}
    hip = C.CDLL(paths.pop())
    draw = DrawParameters(inverse_viewproj=view_along_x().tolist(),
                          camera_position=[0.0, 0.0, 6362.0], sun_direction=[0.6, 0.0, 0.8])
    bufs = [DeviceBuffer(w * h * 16) for _ in range(4)]
    renderer = Renderer(builder)
    renderer.draw(None, a, draw, w, h, bufs[0], bufs[1])
    synchronize()
    s, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(s)) == 0
    relaxed = 2
    assert hip.hipStreamBeginCapture(s, relaxed) == 0
    try:
        print("\n[draw] legacy stream", flush=True)
        renderer.draw(None, a, draw, w, h, bufs[2], bufs[3])
    finally:
        assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0
    synchronize()
    if graph:
        assert hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(s) == 0
    eager_c, eager_t, c, t = (b.to_array(np.float32, (h, w, 4)) for b in bufs)
    a.close()
    assert (rel_err(t, eager_t, 1e-6) > 1e-4).any(-1).mean() < 1e-3
    assert (rel_err(c, eager_c, 1e-4) > 1e-3).any(-1).mean() < 1e-3


@pytest.mark.parametrize("f16", [False, True], ids=["binary32", "binary16"])
@pytest.mark.parametrize("form", ["composite", "composite_no_transmittance", "no_transmittance"])
def test_large_draw_forms_match_fragment_shader(builder, f16, form):
    """The slice draw's other outputs (composited over a background, without a
    transmittance image), on both storage types."""
    w, h = 1500, 1000
    p = Parameters().replace(**DUMP_SIZES, flags=abi.FB_FLAG_F16_STORAGE if f16 else 0)
    pa = Atmosphere.build(builder, None, p)
    pa.wait()
    a = pa.assert_ready()
    T = a.download("transmittance").astype(np.float64)
    S = a.download("scattering").astype(np.float64)
    near = 0.1
    ivp = view_along_x(near)
    draw = DrawParameters(inverse_viewproj=ivp.tolist(), camera_position=[0.0, 0.0, 6362.0],
                          sun_direction=[0.6, 0.0, 0.8])
    rng = np.random.default_rng(5)
    depth = rng.uniform(near / 50e3, near / 500.0, (h, w)).astype(np.float32)
    depth[: h // 2] = 0.0
    back = rng.uniform(0.0, 0.2, (h, w, 4)).astype(np.float32)
    color = DeviceBuffer.from_array(back)
    tr = None if "no_transmittance" in form else DeviceBuffer(w * h * 16)
    print(f"\n[draw] {w}x{h} {form} binary{16 if f16 else 32}", flush=True)
    Renderer(builder).draw(None, a, draw, w, h, color, tr,
                           depth=DeviceBuffer.from_array(depth), composite="composite" in form)
    synchronize()
    g_c = color.to_array(np.float32, (h, w, 4))
    a.close()
    o_c, o_t = Oracle("f32").render_frame(p, T, S, ivp, draw.camera_position,
                                           draw.sun_direction, w, h, depth=depth)
    want = np.asarray(o_c, np.float64)
    if "composite" in form:
        want = want + back * np.asarray(o_t, np.float64)
        assert np.array_equal(g_c[..., 3], back[..., 3])
    else:
        assert np.all(g_c[..., 3] == 0.0)
    assert (rel_err(g_c, want, 1e-4) > 1e-3).any(-1).mean() < 1e-3
    if tr is not None:
        g_t = tr.to_array(np.float32, (h, w, 4))
        assert (rel_err(g_t, o_t, 1e-6) > 1e-4).any(-1).mean() < 1e-3
