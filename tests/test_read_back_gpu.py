"""Read-back of results at the sizes where it changes form (a plain copy, one
piece, several, more than a lane holds) and from several contexts at once:
the bytes are the frame's.  The same channels come through the formatter and
through rh_read_channels, by different kernels."""
import threading

import numpy as np
import pytest

from aqsis_amd import scenes

pytestmark = pytest.mark.gpu


def _hider(res):
    from aqsis_amd.hider import Hider
    opts, prims = scenes.patches_scene(seed=3, n=30, res=res, samples=(1, 1), filt=("box", 1.0, 1.0), size_px=60.0)
    h = Hider(opts)
    h.post_surfaces(prims)
    h.render()
    return h


def _consistent(h):
    ch, rgba = h.channels(), h.rgba8()
    f = h.display_request_values("rgbaz", (0.0, 0.0, 0.0, 0.0), 0, "float32")     # a, r, g, b, z
    assert np.array_equal(f[..., [1, 2, 3, 0, 4]].copy().view(np.uint32), ch[..., [0, 1, 2, 6, 7]].copy().view(np.uint32))
    assert np.array_equal(rgba, h.display_values("uint8"))
    assert np.array_equal(h.channels().view(np.uint32), ch.view(np.uint32))


# bytes of channels: 36 KB, 66 KB, 146 KB, 4.7 MB, 16 MB + 1 row, 54 MB
@pytest.mark.parametrize("res", [(32, 32), (61, 31), (64, 65), (401, 325), (1024, 456), (1500, 1001)])
def test_sizes(res):
    print(f"read back {res}", flush=True)
    h = _hider(res)
    _consistent(h)
    h.close()


def test_contexts_at_once():
    hs = [_hider((401 + 16 * i, 325)) for i in range(6)]
    errs = []

    def work(h):
        try:
            for _ in range(5):
                h.render_device()
                _consistent(h)
        except Exception as e:          # reported by the main thread
            errs.append(e)
    ts = [threading.Thread(target=work, args=(h,)) for h in hs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for h in hs:
        h.close()
    assert not errs, errs
