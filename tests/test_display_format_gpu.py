"""The device's display formatting against the host's (rh_format_display) on
the frame's own channels: every value type, with and without quantisation,
with infinite and NaN channels (negative filter lobes under gamma), values
past every clamp, and one request of each mode."""
import numpy as np
import pytest

from aqsis_amd import scenes
from aqsis_amd.hider import DSPY, format_display, sample_positions

pytestmark = pytest.mark.gpu

QUANTIZE = [(0.0, 0.0, 0.0, 0.0), (255.0, 0.0, 255.0, 0.5), (65535.0, 0.0, 65535.0, 0.5), (127.0, -128.0, 127.0, 0.7),
            (4.0e9, -3.0e9, 5.0e9, 0.5), (1000.0, -40000.0, 40000.0, 0.0)]


@pytest.fixture(scope="module")
def frame():
    from aqsis_amd.hider import Hider
    opts, prims = scenes.patches_scene(seed=5, n=60, res=(53, 41), samples=(2, 2), filt=("bessel", 3.0, 3.0),
                                       size_px=12.0)
    opts.exposure_gamma = 2.2
    opts.num_displays = 2
    for p in prims[::7]:
        p.Cs[:] = [float("inf"), 2.0e5, -3.0]
    print("display formats", flush=True)
    h = Hider(opts)
    h.post_surfaces(prims)
    h.render()
    yield opts, h
    h.close()


@pytest.mark.parametrize("q", QUANTIZE)
@pytest.mark.parametrize("kind", list(DSPY))
def test_values_are_the_hosts(frame, kind, q):
    opts, h = frame
    ch = h.channels()
    assert np.isnan(ch).any() and np.isinf(ch).any()
    one, lo, hi, dither = q
    o = type(opts).from_buffer_copy(opts)
    o.quantize_one, o.quantize_min, o.quantize_max, o.quantize_dither = q
    _, draws = sample_positions(opts, (h.ext_width, h.ext_height, h.spp), (h.width, h.height))
    want = format_display(o, ch, draws, kind)                    # r, g, b, a
    got = h.display_request_values("rgba", q, 0, kind)           # a, r, g, b
    assert np.array_equal(got.view(np.uint8), want[..., [3, 0, 1, 2]].copy().view(np.uint8))
    for index in (0, 1):
        z = h.display_request_values("z", q, index, kind)
        assert z.shape == (h.height, h.width, 1)
    if one == 0.0 and kind == "float32":
        assert np.array_equal(z[..., 0].view(np.uint32), ch[..., 7].copy().view(np.uint32))


@pytest.mark.parametrize("q", QUANTIZE)
@pytest.mark.parametrize("kind", list(DSPY))
def test_depth_requests_of_each_place(oracle, frame, kind, q):
    # depths, the background's FLT_MAX among them (past the 64-bit range when
    # quantised), with the dither draws of each of the two requests
    from aqsis_amd.hider import mode_bits
    opts, h = frame
    ch = h.channels()
    assert (ch[..., 7] == np.finfo(np.float32).max).any()
    for index in (0, 1):
        _, draws = oracle.sample_positions(opts, display=index)
        for mode in ("z", "rgbaz"):
            got = h.display_request_values(mode, q, index, kind)
            want = oracle.display_request_values(q, mode_bits(mode), ch, draws, DSPY[kind])
            assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want).view(np.uint8)), (mode, index)
