"""Performance cases of the hider: frames rendered through `aqsis_amd.hider.Hider`.

A case is one frame shape with one scene, a device layout and the image its
program reads.  `fresh` cases are what a renderer does for every frame of an
animation or a one-off render: surfaces posted, the host split/dice schedule
with occlusion culling, upload, the device frame, the image read back.  The
others render the resident scene again (`Hider.render_device`), as a program
does that keeps a scene and re-renders it, and as bench.py times it.

Scenes are the generators of `aqsis_amd.scenes`: the configurations of
bench.py and of the tests at their sizes, and the same generators at generic
sizes, sample counts and filters.
"""
import math
import random

import numpy as np

from aqsis_amd import scenes
from aqsis_amd.abi import DEPTH_FILTERS
from aqsis_amd.hider import Hider

RGBA_BYTES, CHANNEL_BYTES, Z_BYTES = 4, 36, 4
SURFACE_BYTES = 16 * 3 * 4 + 6 * 4 + 4       # control points, colour, opacity, shading rate


def _case(name, scene, w, h, spp_x, spp_y, filt, fw, n, px, read, **kw):
    c = {"name": name, "scene": scene, "width": w, "height": h, "samples_x": spp_x, "samples_y": spp_y,
         "filter": filt, "filter_width": fw, "surfaces": n, "surface_px": px, "read": read,
         "layout": "grid", "fresh": False}
    c.update(kw)
    return c


def listed():
    return [
        # The smallest call: an icon or material swatch, 16 spheres; launches
        # and waits are all there is.
        _case("swatch_64", "spheres", 64, 64, 4, 4, "gaussian", 2.0, 16, 30.0, "channels"),
        # bench.py's CPU-runnable configuration, rendered again.
        _case("spheres_256", "spheres", 256, 256, 4, 4, "gaussian", 2.0, 64, 30.0, "channels"),
        # The same as a new scene: an animation frame of a small scene.
        _case("spheres_256_new_scene", "spheres", 256, 256, 4, 4, "gaussian", 2.0, 64, 30.0, "rgba8", fresh=True),
        # A preview with the renderer's option defaults (2x2 samples, gaussian
        # 2x2) at a size that is no multiple of the bucket or of a tile.
        _case("preview_637x475", "patches", 637, 475, 2, 2, "gaussian", 2.0, 2500, 21.0, "rgba8"),
        # bench.py's default workload, in the layout its autotuner takes.
        _case("patches_hd", "patches", 1920, 1080, 4, 4, "catmull-rom", 3.0, 10000, 28.0, "rgba8", layout="batched"),
        # The same as a new scene, in the default layout.
        _case("patches_hd_new_scene", "patches", 1920, 1080, 4, 4, "catmull-rom", 3.0, 10000, 28.0, "rgba8",
              fresh=True),
        # bench.py's clustered workload: very uneven buckets, the largest frame.
        _case("clustered_2048", "clustered", 2048, 2048, 4, 4, "gaussian", 2.0, 378000, 16.0, "rgba8",
              layout="batched"),
        # Two frames of the serving stream: transparent surfaces, an ordinary
        # one and a large one at final-quality sampling.
        _case("serving_512", "serving", 512, 512, 4, 4, "gaussian", 2.0, 6000, 7.5, "channels"),
        _case("serving_1024_8x8", "serving", 1024, 1024, 8, 8, "gaussian", 2.0, 12000, 15.0, "rgba8"),
        # bench.py's transparency and motion blur workload.
        _case("motion_256", "motion", 256, 256, 8, 8, "gaussian", 2.0, 600, 28.0, "channels"),
        # Depth of field, an odd frame size and sample count.
        _case("lens_317x211", "dof", 317, 211, 3, 3, "gaussian", 2.0, 900, 28.0, "channels"),
        # A shadow map: the z display with the midpoint depth filter, one box
        # pixel wide, depths read as floats.
        _case("shadow_map_512", "shadow", 512, 512, 2, 2, "box", 1.0, 2000, 20.0, "z"),
    ]


def draw(rng: random.Random):
    """A frame of the same kinds at another size."""
    scene = rng.choice(["spheres", "patches", "patches", "serving", "serving", "motion", "dof", "shadow", "clustered"])
    top = {"spheres": 1024, "patches": 1600, "serving": 1024, "motion": 288, "dof": 480, "shadow": 1024,
           "clustered": 512}[scene]
    low = {"motion": 48, "dof": 64, "clustered": 128}.get(scene, 48)
    side = math.exp(rng.uniform(math.log(low), math.log(top)))
    w = int(side)
    h = max(33, int(side * rng.choice([1.0, 0.75, 9 / 16, 1.0])) + rng.randrange(0, 3))
    if scene == "serving":
        h = w                                  # the stream's frames are square
    k = rng.choice({"motion": [2, 3, 4, 8], "dof": [1, 2, 3, 4], "shadow": [1, 2, 4], "spheres": [1, 2, 3, 4, 8],
                    "patches": [1, 2, 3, 4, 5], "serving": [2, 4, 8], "clustered": [2, 4]}[scene])
    filt, fw = ("gaussian", 2.0)
    if scene in ("spheres", "patches", "dof", "motion"):
        filt, fw = rng.choice([("gaussian", 2.0), ("gaussian", 2.0), ("box", 1.0), ("box", 2.0), ("catmull-rom", 3.0),
                               ("mitchell", 4.0), ("triangle", 2.0), ("sinc", 4.0), ("gaussian", 3.5)])
    elif scene == "shadow":
        filt, fw = "box", 1.0
    if scene == "spheres":
        n, px = int(math.exp(rng.uniform(math.log(4), math.log(300)))), w * 0.12
    elif scene == "serving":
        n, px = rng.randrange(100, 12001), 28.0 * w / 1920.0
    elif scene == "clustered":
        n, px = int(w / 16.0 * h / 16.0 * 23), 16.0
    else:
        px = rng.uniform(8.0, 40.0)
        cover = rng.uniform(0.5, 4.0) if scene != "motion" else rng.uniform(0.5, 5.0)
        n = max(4, min(5000, int(cover * w * h / (px * px))))
    read = "z" if scene == "shadow" else rng.choice(["rgba8", "channels"])
    return _strip(_case("", scene, w, h, k, k, filt, fw, n, px, read, fresh=rng.random() < 0.15,
                 layout=rng.choice(["grid", "batched"])))


def _strip(c):
    return {k: v for k, v in c.items() if k != "name"}


def _scene(c, seed):
    res, spp = (c["width"], c["height"]), (c["samples_x"], c["samples_y"])
    filt = (c["filter"], c["filter_width"], c["filter_width"])
    kind = c["scene"]
    if kind == "spheres":
        return scenes.spheres_scene(seed=seed, n=c["surfaces"], res=res, samples=spp, filt=filt)
    if kind == "serving":
        k = c["surfaces"]
        opts, prims, _ = next(scenes.serving_requests(seed=seed, count=1, sides=(c["width"],), spp=(c["samples_x"],),
                                                      patches=(k, k)))
        return opts, prims
    if kind == "clustered":
        return scenes.clustered_scene(seed=seed, res=res, samples=spp, filt=filt)
    if kind == "motion":
        return scenes.motion_scene(seed=seed, n=c["surfaces"], res=res, size_px=c["surface_px"], samples=spp,
                                   filt=filt)
    opts, prims = scenes.patches_scene(seed=seed, n=c["surfaces"], res=res, size_px=c["surface_px"], samples=spp,
                                       filt=filt)
    if kind == "dof":
        opts.dof[:] = [2.8, 1.2, 16.0]         # the focal plane inside the patches' depth range
    elif kind == "shadow":
        opts.display_z = 1
        opts.depth_filter = DEPTH_FILTERS["midpoint"]
    return opts, scenes.prim_array(prims)


def prepare(case, seed):
    opts, prims = _scene(case, seed)
    if isinstance(prims, list):
        prims = scenes.prim_array(prims)
    h = Hider(opts)
    if case["layout"] == "batched":
        h.set_tuning(mode="batched", split_cost=1 << 18)
    if not case["fresh"]:
        h.post_surfaces(prims)
        h.render()
    return {"hider": h, "prims": prims, "fresh": case["fresh"], "read": case["read"]}


def run(state):
    h = state["hider"]
    if state["fresh"]:
        h.clear_surfaces()
        h.post_surfaces(state["prims"])
        h.render()
    else:
        h.render_device()
    if state["read"] == "rgba8":
        return {"rgba8": h.rgba8()}
    if state["read"] == "z":
        return {"z": h.display_request_values("z")}
    return {"channels": h.channels()}


# Sample tests a micropolygon gets per sample of a pixel, and operations per
# test, as counted by the hider's own counters on the configurations above
# (a moving micropolygon is visited once per part of the shutter).
_TESTS = {"motion": (9.4, 54.0), "dof": (6.0, 60.0)}


def work(case):
    """Surfaces read once, the image written once; the sample tests and the
    filter's multiplications and additions."""
    w, h, ns = case["width"], case["height"], case["samples_x"] * case["samples_y"]
    n, px = case["surfaces"], case["surface_px"]
    mp = n * px * px if case["scene"] != "clustered" else 53.4e6 * (w * h) / 2048.0 ** 2
    per, ops = _TESTS.get(case["scene"], (1.5, 30.0))
    taps = max(1.0, case["filter_width"]) ** 2 * ns
    out = {"rgba8": RGBA_BYTES, "channels": CHANNEL_BYTES, "z": Z_BYTES}[case["read"]]
    return {"bytes": n * SURFACE_BYTES + w * h * out,
            "flops": mp * ns * per * ops + w * h * taps * 7 * 2}


def exact(case, seed):
    """No value: a frame is what the renderer's own 32-bit tests make of its
    jittered samples (which micropolygon of the diced grids is in front at
    each of them, decided by the order and the rounding of those tests), so a
    64-bit rendering is another picture wherever an edge passes a sample.
    Frames are compared bit for bit instead."""
    return None
