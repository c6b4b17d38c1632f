"""The sweeps' plans (which position blocks go to which workgroup, which tiles to which wave) are made on the host.  They are
remembered for every window and number of workgroups: a batch of another size does not throw one away, and those of one window share
what takes longest to make."""
import os
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <memory>
#include <thread>
#include <vector>
#include "dag_chunks.h"
using namespace dagx;
template <int SPACING, int N>
static int check(const ChunkCosts (&costs)[N]) {
    // batches of changing size: every number of workgroups in turn, windows of every number of blocks
    for (int round = 0; round < 2; ++round)
        for (int W = 1; W <= kMaxBlocksFast; ++W) {
            const ChunkPlan<N> *kept[12] = {};
            for (int C = 1; C <= 11; ++C) kept[C] = &chunk_plan<SPACING>(64 * W - 1, C, costs);
            for (int C = 1; C <= 11; ++C) {
                auto fresh = std::make_unique<ChunkPlan<N>>();
                plan_chunks<SPACING>(W, C, costs, *fresh);
                if (std::memcmp(fresh->gtab, kept[C]->gtab, sizeof fresh->gtab) || std::memcmp(fresh->deal, kept[C]->deal, sizeof fresh->deal)) {
                    std::printf("W=%d C=%d: another plan in its place\n", W, C);
                    return 1;
                }
            }
            for (int C = 1; C <= 11; ++C)
                if (kept[C] != &chunk_plan<SPACING>(64 * W, C, costs)) { std::printf("W=%d C=%d: made again\n", W, C); return 1; }
        }
    // a window longer than any graph the sweeps take is that of the longest
    return &chunk_plan<SPACING>(8192, 4, costs) != &chunk_plan<SPACING>(64 * kMaxBlocksFast, 4, costs);
}
// us to make the plans of a window for C = 1 .. most, on a thread that has made none: the median of 41
static double first(const ChunkCosts (&costs)[2], int translen, int most) {
    std::vector<double> us;
    for (int round = 0; round < 41; ++round)
        std::thread([&] {
            const auto start = std::chrono::steady_clock::now();
            for (int C = 1; C <= most; ++C) chunk_plan<1>(translen, C, costs);
            us.push_back(std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - start).count());
        }).join();
    std::sort(us.begin(), us.end());
    return us[20];
}
int main() {
    static const ChunkCosts loss[2] = {{45, 7, 4, 100}, {85, 17, 11, 100}}, one[1] = {{62, 27, 4, 75}}, two[1] = {{36, 27, 4, 75}};
    // eleven plans, as the first loss call of a window may weigh: each for itself they took eleven times as long as one
    for (const int translen : {300, 511, 1023})
        if (first(loss, translen, 11) > 7 * first(loss, translen, 1)) { std::printf("translen %d: %.0f us, one plan %.0f us\n", translen, first(loss, translen, 11), first(loss, translen, 1)); return 1; }
    return check<1>(loss) || check<1>(one) || check<2>(two);
}
"""


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
def test_a_plan_outlives_calls_with_other_numbers_of_workgroups(tmp_path):
    src, exe = tmp_path / "plans.hip", tmp_path / "plans"
    src.write_text(PROGRAM)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-function",
                    "-pthread", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "da_transformer_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
