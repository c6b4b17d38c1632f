"""The sweeps' plans (which position blocks go to which workgroup, which tiles to which wave) are made on the host.  They are
remembered for every window and number of workgroups: a batch of another size does not throw one away, and those of one window share
what takes longest to make."""
import os
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <memory>
#include <vector>
#include "dag_chunks.h"
using namespace dagx;
template <int SPACING, int N, typename COSTS>
static int check(COSTS costs_of) {
    // batches of changing size: every number of workgroups in turn, windows of every number of blocks
    for (int round = 0; round < 2; ++round)
        for (int W = 1; W <= kMaxBlocksFast; ++W) {
            const ChunkCosts (&costs)[N] = costs_of(64 * W);
            const ChunkPlan<N> *kept[12] = {};
            for (int C = 1; C <= 11; ++C) kept[C] = &chunk_plan<SPACING>(64 * W - 1, C, costs);
            for (int C = 1; C <= 11; ++C) {
                auto fresh = std::make_unique<ChunkPlan<N>>();
                plan_chunks<SPACING>(W, C, costs, *fresh);
                if (std::memcmp(fresh->gtab, kept[C]->gtab, sizeof fresh->gtab) || std::memcmp(fresh->deal, kept[C]->deal, sizeof fresh->deal) ||
                    std::memcmp(fresh->busiest, kept[C]->busiest, sizeof fresh->busiest)) {
                    std::printf("W=%d C=%d: another plan in its place\n", W, C);
                    return 1;
                }
            }
            if (&group_deals<SPACING>(64 * W - 1, costs) != &group_deals<SPACING>(64 * W, costs)) { std::printf("W=%d: deals made again\n", W); return 1; }
            for (int C = 1; C <= 11; ++C)
                if (kept[C] != &chunk_plan<SPACING>(64 * W, C, costs)) { std::printf("W=%d C=%d: made again\n", W, C); return 1; }
        }
    // a window longer than any graph the sweeps take is that of the longest
    return &chunk_plan<SPACING>(8192, 4, costs_of(8192)) != &chunk_plan<SPACING>(64 * kMaxBlocksFast, 4, costs_of(8192));
}
// blocks of the groups of a graph of nb blocks
template <int SPACING>
static bool groups_are(const ChunkCosts &cost, int W, int C, int nb, std::vector<int> want) {
    const ChunkCosts costs[1] = {cost};
    ChunkPlan<1> plan;
    plan_chunks<SPACING>(W, C, costs, plan);
    std::vector<int> got;
    for (int q = 0; q < C && plan.gtab[0][nb][q + 1] > plan.gtab[0][nb][q]; ++q) got.push_back(plan.gtab[0][nb][q + 1] - plan.gtab[0][nb][q]);
    if (got == want) return true;
    std::printf("W=%d C=%d nb=%d:", W, C, nb);
    for (const int n : got) std::printf(" %d", n);
    std::printf("\n");
    return false;
}
// Every group of an alignment's plan has its tiles and foreign blocks dealt to waves that have room for them, and fits a CU's LDS: one that
// does not sends its samples to the one-workgroup redo.
template <int SPACING>
static bool alignment_fits(int B, int T, int L, int translen, int C) {
    const ChunkPlan<1> &plan = chunk_plan<SPACING>(translen, C, align_costs<SPACING>(translen));
    const int W = (translen + kBlk - 1) / kBlk;
    for (int nb = 1; nb <= (L + kBlk - 1) / kBlk; ++nb) {
        const unsigned char *g = plan.gtab[0][nb];
        int n = 0;
        bool ok = plan.busiest[0][nb] < kNoPlan;
        for (int q = 0; q < C; ++q) {
            if (g[q + 1] == g[q]) continue;
            const int size = g[q + 1] - g[q];
            int tiles = 0, foreign = 0, want = 0;
            ok = ok && q == n++ && size > 0 && size <= kChunkBlocks;
            for (int w = 0; ok && w < kTileWaves; ++w) {
                const int mine = dealt_tiles(plan.deal[0][nb][q], w), fetch = dealt_foreign(plan.deal[0][nb][q], w);
                ok = w >= size || (mine <= SPACING && (fetch == 0 || size == kTileWaves));
                tiles += mine; foreign += fetch;
            }
            for (int J = g[q]; J < g[q + 1]; ++J) want += tiles_of_block<SPACING>(J, W);
            ok = ok && tiles == want && foreign == g[q] - tile_ilo(g[q], W) && align_lds(g[q], size, W, SPACING).total * 4 <= kChunkLdsBytes;
        }
        if (ok && g[0] == 0 && g[n] == nb) continue;
        std::printf("alignment B=%d T=%d L=%d translen=%d: C=%d nb=%d\n", B, T, L, translen, C, nb);
        return false;
    }
    return true;
}
static int alignment() {
    int seen = 0;
    for (int B = 1; B <= 128; B += B < 70 ? 3 : 29)
        for (int L = 2; L <= 1024; L += 31)
            for (int translen = 1; translen < L; translen = translen < 64 ? 64 : translen + 64) {
                const int T = L;
                if (!align_in_chunks(B, T, L, translen)) continue;
                const int C = align_groups(B, T, L, translen);
                if (C == 0) continue;
                ++seen;
                if (align_spacing((L + kBlk - 1) / kBlk, C) == 2 ? !alignment_fits<2>(B, T, L, translen, C) : !alignment_fits<1>(B, T, L, translen, C)) return 1;
            }
    return seen < 3000;
}
// where the alignment's sweep goes in chunks: the step at which it begins to
static bool chunks_from(int B, int L, int translen, int T) {
    if (!align_in_chunks(B, T - 1, L, translen) && align_in_chunks(B, T, L, translen)) return true;
    std::printf("alignment B=%d L=%d translen=%d: not in chunks from T=%d on\n", B, L, translen, T);
    return false;
}
int main() {
    // (eight blocks with a workgroup each, and with less room; other graphs; windows of at most three blocks)
    if (!chunks_from(1, 449, 448, 43) || !chunks_from(32, 512, 193, 43) || !chunks_from(33, 512, 511, 38) || !chunks_from(32, 448, 447, 36) ||
        !chunks_from(32, 513, 512, 40) || !chunks_from(32, 512, 192, 46) || !chunks_from(1, 1024, 1023, 54) || !chunks_from(64, 192, 191, 26)) return 1;
    // groupings as good as each other for the busiest SIMD: more even ones, where they gain more than their hand-overs take
    if (!groups_are<2>(align_costs<2>(64)[0], 1, 8, 8, {2, 2, 2, 2}) || !groups_are<1>(align_costs<1>(192)[0], 3, 10, 13, {3, 2, 2, 2, 2, 2}) ||
        !groups_are<1>(kSweepCosts[0], 5, 2, 5, {3, 2}) || !groups_are<1>(align_costs<1>(576)[0], 9, 9, 9, {4, 2, 1, 1, 1}) ||
        !groups_are<2>(align_costs<2>(128)[0], 2, 8, 8, {3, 2, 2, 1}) || !groups_are<1>(align_costs<1>(128)[0], 2, 2, 14, {8, 6}) ||
        !groups_are<1>(align_costs<1>(896)[0], 14, 10, 14, {4, 2, 1, 1, 1, 1, 1, 1, 1, 1})) return 1;
    return check<1, 2>([](int) -> const ChunkCosts (&)[2] { return kSweepCosts; }) || check<1, 1>(align_costs<1>) || check<2, 1>(align_costs<2>) || alignment();
}
"""


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
def test_a_plan_outlives_calls_with_other_numbers_of_workgroups(tmp_path):
    src, exe = tmp_path / "plans.hip", tmp_path / "plans"
    src.write_text(PROGRAM)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-function",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "da_transformer_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
