"""The library's host side on a HIP runtime that runs on the CPU (fake_hip.cpp).
Reading results back: where its memory comes from and how long it is kept, what
it waits for and what it holds meanwhile, and what a failed copy leaves behind.
The estimate of a frame's device memory against what a context takes.  The
growth of the transparent-hit arena at its limits.  Each case is a process of its own; its frames hold no surfaces, so their
channels are what the fake's new memory holds."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/include"

PRELUDE = """
import ctypes as C, sys, threading, time
sys.path.insert(0, sys.argv[2])
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_held.restype = C.c_uint64
fake.fake_most.argtypes = [C.c_uint64]
import numpy as np
from aqsis_amd import hider, scenes
from aqsis_amd.abi import default_options

def rendered(w, h):
    x = hider.Hider(default_options(xres=w, yres=h, filter="box", filter_xwidth=1.0, filter_ywidth=1.0))
    x.render()
    return x

def right(a):
    v = a.reshape(-1).view(np.uint32)
    return np.array_equal(v, (np.arange(v.size, dtype=np.uint64) * 2654435761).astype(np.uint32))

LANE, SLAB = 17 << 20, 64 << 10
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists(os.path.join(HIP, "hip", "hip_runtime_api.h")):
        pytest.skip("g++ or the HIP headers are not installed")
    d = tmp_path_factory.mktemp("fake")
    so = str(d / "libfake.so")
    subprocess.run([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", HIP,
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so, "-lpthread"], check=True)

    def go(code):
        src = d / "case.py"
        src.write_text(PRELUDE + textwrap.dedent(code))
        r = subprocess.run([sys.executable, str(src), so, ROOT], capture_output=True, text=True, timeout=90)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


def test_sizes_and_devices(run):
    # a context on device 1, read while device 0 is current: whole results,
    # and nothing is allocated on the device that is only current
    run("""
    for size in ((32, 32), (61, 31), (64, 65), (401, 325), (1024, 456), (1500, 1001)):
        fake.hipSetDevice(1)
        h = rendered(*size)
        fake.hipSetDevice(0)
        assert right(h.channels()) and right(h.rgba8()), size
        assert fake.fake_held(0) == 0, size
        h.close()
    """)


def test_failed_copy_leaves_nothing(run):
    # a stream that ends without the data gives an error, and the next copy is whole
    run("""
    h = rendered(401, 325)
    fake.fake_lose(1)
    try:
        h.channels()
        raise SystemExit("no error")
    except hider.HiderError:
        pass
    fake.fake_lose(0)
    for _ in range(3):
        assert right(h.channels())
    """)


def test_a_context_a_frame(run):
    # contexts one after another take pinned memory once, and never wait for the device
    run("""
    calls = []
    for _ in range(6):
        h = rendered(256, 256)
        assert right(h.rgba8()) and right(h.channels())
        h.close()
        calls.append(fake.fake_pinned_calls())
    assert calls[0] > 0 and calls == [calls[0]] * 6, calls
    assert fake.fake_device_syncs() == 0
    """)


def test_pinned_memory_is_bounded_and_handed_back(run):
    # many contexts read at once on four lanes at most; with the last of them
    # all goes back but one lane and one slab of counter blocks
    run("""
    for _ in range(2):
        hs = [rendered(401, 325) for _ in range(12)]
        small = [rendered(16, 16) for _ in range(600)]
        ok = [True] * len(hs)
        def work(i):
            for _ in range(4):
                ok[i] = ok[i] and right(hs[i].channels())
        ts = [threading.Thread(target=work, args=(i,)) for i in range(len(hs))]
        fake.fake_gate(0)
        for t in ts: t.start()
        while fake.fake_waiting() < 4: time.sleep(0.01)
        fake.fake_gate(-1)
        for t in ts: t.join()
        assert all(ok)
        assert 4 * (16 << 20) <= fake.fake_held(-1) <= 4 * LANE + 4 * SLAB
        for h in hs + small: h.close()
        assert fake.fake_held(-1) <= LANE + SLAB, fake.fake_held(-1)
    """)


@pytest.mark.parametrize("workgroups", [0, 1, 9, 37])
def test_other_threads_have_the_worker_pool(run, workgroups):
    # a read whose data has not come, or only its first parts, does not keep a
    # schedule of another thread from the worker pool
    run("""
    opts, prims = scenes.patches_scene(seed=1, n=400, res=(320, 240))
    h = rendered(1024, 456)
    out = []
    fake.fake_gate(%d)
    a = threading.Thread(target=lambda: out.append(right(h.channels())), daemon=True)
    a.start()
    while fake.fake_waiting() < 1: time.sleep(0.01)
    time.sleep(0.05)
    b = threading.Thread(target=lambda: hider.estimate(opts, prims), daemon=True)
    b.start()
    b.join(20)
    assert not b.is_alive(), "the schedule waits for the read"
    assert a.is_alive()
    fake.fake_gate(-1)
    a.join()
    assert out == [True]
    """ % workgroups)


def test_without_pinned_memory(run):
    # the driver refuses pinned memory: contexts are made and frames read by plain copies
    run("""
    fake.fake_refuse_pinned(1)
    for _ in range(2):
        h = rendered(401, 325)
        assert right(h.channels()) and right(h.rgba8())
        h.render_device()
        h.render_device_noalloc()
        assert h.stats()["spl_count"] == 0
        h.close()
    fake.fake_refuse_pinned(0)
    h, g = rendered(401, 325), rendered(64, 64)
    assert right(h.channels())
    h.close(); g.close()
    assert fake.fake_held(-1) == LANE // 17 * 16 + 4096 + SLAB
    """)


@pytest.mark.parametrize("samples", [(1, 1), (2, 2), (3, 3), (4, 4), (8, 8)])
def test_estimate_holds_what_a_context_takes(run, samples):
    # with even filter widths the box tests may differ between pixels and are
    # kept by pixel; a job admitted by its estimate has to have room for them
    run("""
    for res in ((48, 40), (256, 256), (637, 475)):
        for width, varies in ((1.0, 0), (2.0, 1), (2.5, 0), (3.0, 0), (4.0, 1), (6.0, 1), (7.0, 0)):
            for bucket, lens in ((16, 0), (32, 0), (16, 1)):
                if res[0] > 256 and (bucket != 32 or width not in (1.0, 4.0)): continue
                o = default_options(xres=res[0], yres=res[1], xsamples=%d, ysamples=%d, filter="gaussian",
                                    filter_xwidth=width, filter_ywidth=width)
                o.bucket_x = o.bucket_y = bucket
                if lens: o.dof[:] = [22.0, 45.0, 1200.0]
                fake.fake_box_varies(varies)
                h = hider.Hider(o)
                h.render()
                need, said = fake.fake_held(0), hider.estimate(o, [])["device_bytes"]
                h.close()
                assert need <= said, (res, width, bucket, lens, need, said)
                # (the tests' room is kept for frames that take tiles, too)
                assert varies or said <= need + need // 20 + (256 << 10), (res, width, bucket, lens, need, said)
    """ % samples)


@pytest.mark.parametrize("missing,taken", [(1 << 20, True), (1_600_000_000, True), (1_900_000_000, True),
                                           (2_146_000_000, True), (2_147_483_647, False)])
def test_arena_grows_to_its_limit(run, missing, taken):
    # entries below 2^31 in all: the spare quarter does not count against them
    run("""
    h = hider.Hider(default_options(xres=64, yres=64))
    fake.fake_no_room(%d)
    try:
        h.render()
        assert %r
    except hider.HiderError as e:
        assert not %r and "2^31" in str(e), e
    """ % (missing, taken, taken))


def test_no_frame_on_an_arena_that_could_not_grow(run):
    run("""
    h = hider.Hider(default_options(xres=64, yres=64))
    h.render()
    for again in (h.render_device, h.render_device_noalloc, h.render_stages):
        fake.fake_no_room(1 << 22)
        fake.fake_most(1 << 20)
        for f in (h.render_device, again):
            try:
                f()
                raise SystemExit("a frame on a missing arena")
            except hider.HiderError:
                pass
        fake.fake_most(1 << 40)
        h.render()
        again()
    """)


def test_results_come_by_the_kernel(run):
    # results of every size by way of a lane: no copy by the runtime, and no wait
    # for the stream once all parts are there
    run("""
    for size in ((1, 1), (16, 16), (48, 44), (160, 120), (401, 325)):
        h = rendered(*size)
        for read in (h.channels, h.rgba8):
            before = fake.fake_plain_copies(), fake.fake_pinned_copies(), fake.fake_stream_waits()
            assert right(read())
            assert (fake.fake_plain_copies(), fake.fake_pinned_copies(), fake.fake_stream_waits()) == before
        h.close()
    """)
