"""The lens sampler's split of a task over workgroups and its 8x8-pixel tasks:
one to sixty-four lens cells, frames that end inside a tile, buckets narrower
and wider than a task; every output and counter the oracle's."""
import numpy as np
import pytest

from aqsis_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bucket", [(16, 16), (32, 8), (6, 40)])
@pytest.mark.parametrize("k", [(1, 1), (2, 2), (3, 3), (5, 3), (8, 8)])
def test_lens_cells(oracle, k, bucket):
    from aqsis_amd.hider import Hider
    print(f"lens {k} bucket {bucket}", flush=True)
    opts, prims = scenes.patches_scene(seed=11, n=70, res=(67, 45), samples=k, filt=("gaussian", 2.0, 2.0),
                                       size_px=14.0, opacity=(0.4, 1.0))
    for p in prims[::2]:
        p.Os[:] = [1.0, 1.0, 1.0]
    opts.bucket_x, opts.bucket_y = bucket
    opts.dof[:] = [2.8, 1.2, 16.0]
    ref = oracle.render(opts, prims, occlusion_cull=True)
    with Hider(opts) as h:
        h.post_surfaces(prims)
        h.render()
        ids, depth, rgbaz = h.samples()
        st = h.stats()
        ch = h.channels()
    assert np.array_equal(ids, ref["mp_id"])
    assert np.array_equal(depth.view(np.uint32), ref["depth"].view(np.uint32))
    assert np.array_equal(rgbaz.view(np.uint32), ref["rgbaz"].view(np.uint32))
    assert np.array_equal(ch.view(np.uint32), ref["channels"].view(np.uint32))
    for key in ("spl_count", "spl_bound_hits", "spl_hits"):
        assert st[key] == ref["stats"][key], key


# With 1 or 2 samples a pixel a task is 2 or 4 tiles where 1024 tasks are left:
# frames on both sides of the lines, wide buckets, a crop window.
@pytest.mark.parametrize("k,res,bucket,crop", [((1, 1), (380, 340), (16, 16), None), ((1, 1), (400, 330), (16, 16), None),
                                               ((2, 1), (400, 330), (32, 32), None), ((1, 2), (401, 333), (16, 16), None),
                                               ((1, 1), (520, 521), (16, 16), None),
                                               ((1, 1), (600, 600), (24, 16), (0.04, 0.96, 0.03, 0.97))])
def test_lens_tasks_of_more_tiles(oracle, k, res, bucket, crop):
    from aqsis_amd.hider import Hider
    print(f"lens {k} {res} bucket {bucket}", flush=True)
    opts, prims = scenes.patches_scene(seed=12, n=60, res=res, samples=k, filt=("gaussian", 2.0, 2.0), size_px=60.0,
                                       opacity=(0.4, 1.0), shading_rate=4.0)
    for p in prims[::2]:
        p.Os[:] = [1.0, 1.0, 1.0]
    opts.bucket_x, opts.bucket_y = bucket
    opts.dof[:] = [2.8, 1.2, 16.0]
    if crop:
        opts.crop[:] = crop
    ref = oracle.render(opts, prims, occlusion_cull=True)
    with Hider(opts) as h:
        h.post_surfaces(prims)
        h.render()
        h.render_device_noalloc()
        ids, depth, rgbaz = h.samples()
        st = h.stats()
        ch = h.channels()
    assert np.array_equal(ids, ref["mp_id"])
    assert np.array_equal(depth.view(np.uint32), ref["depth"].view(np.uint32))
    assert np.array_equal(rgbaz.view(np.uint32), ref["rgbaz"].view(np.uint32))
    assert np.array_equal(ch.view(np.uint32), ref["channels"].view(np.uint32))
    for key in ("spl_count", "spl_bound_hits", "spl_hits"):
        assert st[key] == ref["stats"][key], key
