"""How a frame is cut into sampling tasks: the finer cuts (8x8-pixel tasks of
wide blocks and of lens frames) never make a frame outgrow the counter rows of
rh_render_device_noalloc that the coarse cut (parts of four blocks a side)
fits, frames of ordinary size keep them, and the tasks cover the sampled
region once.  Host code only, compiled here."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "aqsis_amd", "csrc")

HARNESS = r'''
#include "front.h"
#include <algorithm>
#include <cfloat>
#include <cstdio>
#include <string>
// stdin: cases of  xres yres bucket xs ys lens; stdout: per case the tasks,
// those of the coarse cut, and whether the tasks cover the region once
int main() {
    int xres, yres, bucket, xs, ys, lens;
    while (std::scanf("%d %d %d %d %d %d", &xres, &yres, &bucket, &xs, &ys, &lens) == 6) {
        rh_options o = {};
        o.xres = xres; o.yres = yres; o.pixel_aspect = 1.0f;
        o.crop[1] = o.crop[3] = 1.0f;
        o.fov = 45.0f; o.clip_near = FLT_EPSILON; o.clip_far = FLT_MAX;
        o.xsamples = xs; o.ysamples = ys;
        o.filter = RH_FILTER_GAUSSIAN; o.filter_xwidth = o.filter_ywidth = 2.0f;
        o.bucket_x = o.bucket_y = bucket;
        o.dof[0] = lens ? 22.0f : FLT_MAX;
        o.dof[1] = 45.0f; o.dof[2] = 1200.0f;
        rh::Shape s;
        std::string err;
        if (!rh::make_shape(o, s, err)) { std::printf("refused %s\n", err.c_str()); return 1; }
        long coarse = 0, area = 0;
        bool ok = true;
        for (size_t k = 0; k < s.buckets.size(); ++k) {
            const auto& b = s.buckets[k];
            const int ow = b.sx1 - b.sx0, oh = b.sy1 - b.sy0;
            if (ow > 0 && oh > 0)
                coarse += std::min(ow, std::max(1, std::min(4, bucket / (4 * s.blockW)))) *
                          std::min(oh, std::max(1, std::min(4, bucket / (4 * s.blockH))));
            int y = b.sy0;
            for (int t = s.taskStart[k]; t < s.taskStart[k + 1];) {
                int x = b.sx0;
                const int y1 = s.tasks[t].y1;
                for (; t < s.taskStart[k + 1] && s.tasks[t].y0 == y; ++t) {
                    const auto& T = s.tasks[t];
                    ok = ok && T.bucket == (int)k && T.x0 == x && T.x1 > T.x0 && T.y1 == y1 && y1 > y;
                    x = T.x1;
                    area += (long)(T.x1 - T.x0) * (T.y1 - T.y0);
                }
                ok = ok && x == b.sx1;
                y = y1;
            }
            ok = ok && (ow <= 0 || oh <= 0 || y == b.sy1);
        }
        ok = ok && area == (long)s.extW * s.extH;
        std::printf("%zu %ld %d\n", s.tasks.size(), coarse, ok ? 1 : 0);
    }
    return 0;
}
'''

ROWS = ((4 << 20) - 256) // 20            # counter rows the no-allocation form holds


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not installed")
    d = tmp_path_factory.mktemp("tasks")
    src = d / "h.cpp"
    src.write_text(HARNESS)
    exe = d / "h"
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC, str(src),
                    os.path.join(CSRC, "front.cpp"), "-o", str(exe), "-lpthread"], check=True)

    def run(cases):
        text = "\n".join(" ".join(str(int(v)) for v in c) for c in cases)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
        return [tuple(int(v) for v in line.split()) for line in out[:len(cases)]]
    return run


@pytest.mark.parametrize("lens", [0, 1])
@pytest.mark.parametrize("samples", [(1, 1), (2, 2), (3, 3), (4, 4), (8, 8)])
def test_no_finer_than_the_counter_rows(split, samples, lens):
    cases = [(res, res, bucket, *samples, lens)
             for bucket in (16, 24, 32, 48, 64) for res in (1024, 2048, 3000, 3840, 4096, 6144, 8192)]
    for case, (tasks, coarse, ok) in zip(cases, split(cases)):
        assert ok, case
        up = (tasks + 127) // 128 * 128            # the launches round up
        if (coarse + 127) // 128 * 128 <= ROWS:
            assert up <= ROWS, (case, tasks, coarse)


def test_ordinary_frames_keep_the_finer_cut(split):
    # 8x8 pixels a task
    for case, (tasks, coarse, ok) in [((2048, 2048, 16, 2, 2, 0), (65536, 16384, 1)),
                                      ((640, 480, 32, 2, 2, 0), (20 * 15 * 16, 20 * 15 * 4, 1))]:
        assert split([case]) == [(tasks, coarse, ok)]
