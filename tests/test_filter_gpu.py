"""The filter kernels at the shapes where they change form: filter widths from
one pixel to seven (1 to 7 columns and rows),
sample counts on both sides of 32 and odd ones under even
widths (box tests that vary between pixels), frames that are no multiple of a
strip, gamma, and values that are infinite.  The filter sums in the
reference's order, so channels are the oracle's bit for bit (NaNs by position:
the default NaN's sign is the hardware's)."""
import numpy as np
import pytest

from aqsis_amd import scenes

pytestmark = pytest.mark.gpu


def _check(oracle, opts, prims):
    from aqsis_amd.hider import Hider
    ref = oracle.render(opts, prims, occlusion_cull=True)
    with Hider(opts) as h:
        h.post_surfaces(prims)
        h.render()
        ch, rgba = h.channels(), h.rgba8()
    nan = np.isnan(ref["channels"])
    assert np.array_equal(nan, np.isnan(ch))
    assert np.array_equal(ch[~nan].view(np.uint32), ref["channels"][~nan].view(np.uint32))
    assert np.array_equal(rgba, ref["rgba8"])


def _scene(res, k, filt, w, n=40, **kw):
    return scenes.patches_scene(seed=7, n=n, res=res, samples=(k, k), filt=(filt, w, w), size_px=14.0, **kw)


@pytest.mark.parametrize("k", [1, 2, 3, 5, 6, 8])
@pytest.mark.parametrize("filt,w", [("box", 1.0), ("gaussian", 2.0), ("catmull-rom", 3.0), ("gaussian", 3.5),
                                    ("sinc", 4.0), ("triangle", 5.0), ("bessel", 7.0)])
def test_widths_and_samples(oracle, filt, w, k):
    print(f"filter {filt} {w} samples {k}x{k}", flush=True)
    _check(oracle, *_scene((61, 35), k, filt, w))


@pytest.mark.parametrize("res", [(8, 8), (9, 33), (200, 31), (7, 130)])
def test_ragged_frames(oracle, res):
    print(f"frame {res}", flush=True)
    _check(oracle, *_scene(res, 4, "gaussian", 2.0))


@pytest.mark.parametrize("wx,wy", [(1.0, 4.0), (5.0, 2.0), (7.0, 1.0)])
def test_unequal_widths_with_gamma(oracle, wx, wy):
    print(f"widths {wx} {wy}", flush=True)
    opts, prims = _scene((50, 44), 3, "gaussian", 2.0)
    opts.filter_xwidth, opts.filter_ywidth = wx, wy
    opts.exposure_gain, opts.exposure_gamma = 1.3, 2.2
    _check(oracle, opts, prims)


@pytest.mark.parametrize("k", [4, 8])
@pytest.mark.parametrize("filt,w", [("gaussian", 2.0), ("catmull-rom", 3.0)])
def test_infinite_values(oracle, filt, w, k):
    print(f"infinite colours {filt} {k}x{k}", flush=True)
    opts, prims = _scene((64, 40), k, filt, w)
    for p in prims[::9]:
        p.Cs[:] = [float("inf"), 1.0, -float("inf")]
    _check(oracle, opts, prims)


# Even widths with an odd number of samples a side take 8x8-pixel tiles up to a
# size: tiles cut by the frame's edge, crop windows, gamma, infinities, and the
# last frame with tiles beside the first without.
@pytest.mark.parametrize("res", [(8, 8), (9, 33), (200, 31), (7, 130), (64, 40)])
@pytest.mark.parametrize("samples,w", [((3, 3), 2.0), ((3, 3), 4.0), ((1, 1), 4.0), ((2, 1), 6.0), ((1, 2), 6.0)])
def test_tiled_frames(oracle, res, samples, w):
    print(f"tiles {res} {samples} {w}", flush=True)
    opts, prims = scenes.patches_scene(seed=9, n=40, res=res, samples=samples, filt=("catmull-rom", w, w), size_px=14.0)
    for p in prims:
        p.no_cull_hidden = 1          # a frame of one column of buckets may have no culling schedule
    _check(oracle, opts, prims)


@pytest.mark.parametrize("wx,wy,gamma", [(2.0, 4.0, 1.0), (4.0, 1.0, 2.2), (6.0, 2.5, 2.2), (4.0, 4.0, 1.0)])
def test_tiled_crops(oracle, wx, wy, gamma):
    print(f"tiles cropped {wx} {wy} {gamma}", flush=True)
    opts, prims = scenes.patches_scene(seed=9, n=40, res=(90, 70), samples=(1, 3), filt=("gaussian", wx, wy), size_px=14.0)
    opts.crop[:] = [0.13, 0.87, 0.21, 0.93]
    opts.exposure_gamma = gamma
    _check(oracle, opts, prims)


@pytest.mark.parametrize("samples,w", [((3, 3), 2.0), ((1, 1), 4.0)])
def test_tiled_infinite_values(oracle, samples, w):
    print(f"tiles infinite colours {samples} {w}", flush=True)
    opts, prims = scenes.patches_scene(seed=9, n=40, res=(64, 40), samples=samples, filt=("gaussian", w, w), size_px=14.0)
    for p in prims[::9]:
        p.Cs[:] = [float("inf"), 1.0, -float("inf")]
    _check(oracle, opts, prims)


@pytest.mark.parametrize("res", [(316, 316), (317, 316)])
def test_tiled_and_first_without(oracle, res):
    print(f"tiles up to 100000 pixels {res}", flush=True)
    _check(oracle, *scenes.patches_scene(seed=9, n=12, res=res, samples=(4, 3), filt=("gaussian", 2.0, 2.0), size_px=60.0))
