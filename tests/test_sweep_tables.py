"""A sweep launch may choose between tables that give long samples more workgroups and short ones fewer.  Whatever it chooses, every
group of every sample has exactly one workgroup, no group comes in front of the ones it waits for, and a group's tiles and
foreign blocks are all dealt to waves that have room for them."""
import os
import subprocess

import pytest

from conftest import ROOT
from test_gpu_dag_chunks import TABLE_BATCHES, mixed_lengths, table_lengths

PROGRAM = r"""
#include <cstdio>
#include <random>
#include <set>
#include <tuple>
#include "dag_chunks.h"
using namespace dagx;
static int fail(const char *what, int B, int T, int L, int W, int x) { std::printf("%s: B=%d T=%d L=%d translen=%d table %d\n", what, B, T, L, W, x); return 1; }
int main() {
    std::mt19937 rng(5);
    auto draw = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    int offered = 0, chosen = 0;
    const auto tables_of = [](const int B, const int T, const int L, const int which) {
        static GroupTable some[kMostTables];
        TableChoice choice;
        make_tables<1>(some, choice, B, T, L, L - 1, sweep_groups(B, L, L - 1), kMaxGroups, kSweepCosts, which);
        return choice.ntable;
    };
    // a bound that is hardly above a walk's own length is left alone
    if (tables_of(32, 256, 512, 0) != 1 || tables_of(13, 157, 458, 0) != 1 || tables_of(16, 256, 1024, 0) == 1 || tables_of(32, 162, 554, 0) == 1) return fail("offers", 32, 256, 512, 511, 0);
    static GroupTable tables[kMostTables];
    TableChoice t;
    for (int round = 0; round < 3000; ++round) {
        const int B = draw(1, 70), L = draw(1, 1024), T = draw(1, L < 300 ? L : 300), W = draw(0, 1) ? L : draw(1, L);
        const int least = sweep_groups(B, L, W);
        if (least == 0) continue;
        const int which = round & 1, NB = (L + kBlk - 1) / kBlk, blocks = (W + kBlk - 1) / kBlk;
        const int room = draw(0, 2) ? kMaxGroups : draw(least, kMaxGroups);   // groups a sweep that the workspace has words for
        make_tables<1>(tables, t, B, T, L, W, least, room, kSweepCosts, which);
        if (t.ntable < 1 || t.ntable > kMostTables || t.most < least || t.most > kMaxGroups || t.least != least) return fail("sizes", B, T, L, W, 0);
        if (t.most > room) return fail("more groups than the workspace has", B, T, L, W, 0);
        offered += t.ntable > 1;
        for (int x = 0; x < t.ntable; ++x)
            for (int nb = 1; nb <= NB; ++nb) {
                const unsigned char *g = tables[x].gtab[nb];
                int n = 0;
                for (int q = 0; q < kMaxGroups; ++q) {
                    if (g[q + 1] < g[q]) return fail("order", B, T, L, W, x);
                    if (g[q + 1] == g[q]) continue;
                    if (q != n) return fail("an empty group in between", B, T, L, W, x);
                    ++n;
                    const int size = g[q + 1] - g[q], lds = chunk_lds(g[q], size, blocks, which != 0).total * 4;
                    int tiles = 0, foreign = 0, want = 0;
                    for (int w = 0; w < kTileWaves; ++w) {
                        const int mine = dealt_tiles(tables[x].deal[nb][q], w), fetch = dealt_foreign(tables[x].deal[nb][q], w);
                        if (w < size && (mine > 1 || (fetch > 0 && size < kTileWaves))) return fail("a walking wave's room", B, T, L, W, x);
                        tiles += mine; foreign += fetch;
                    }
                    for (int J = g[q]; J < g[q + 1]; ++J) want += tiles_of_block<1>(J, blocks);
                    if (size > kChunkBlocks || tiles != want || foreign != g[q] - tile_ilo(g[q], blocks) || lds > kChunkLdsBytes) return fail("a group", B, T, L, W, x);
                }
                if (g[0] != 0 || g[n] != nb) return fail("cover", B, T, L, W, x);
                if (x > 0 && n != (int)(t.ngroups[x] >> (4 * (nb - 1)) & 15)) return fail("number of groups", B, T, L, W, x);
            }
        // what a launch does with lengths between `low` and L
        const int low = draw(0, 2) ? 3 * L / 4 : draw(0, L);
        int groups[64];
        for (int x = t.ntable - 1; x > 0; --x) {
            int all = 0;
            for (int b = 0; b < B; ++b) {
                const int len = draw(low, L), nb = len >= 1 ? (len + kBlk - 1) / kBlk : 1;
                groups[b] = (int)(t.ngroups[x] >> (4 * (nb - 1))) & 15;
                if (groups[b] < 1) return fail("a sample without a group", B, T, L, W, x);
                all += 2 * groups[b];
            }
            if (all > 2 * ((B + 7) & ~7) * t.most) return fail("more workgroups than the grid has", B, T, L, W, x);
            if (all > kSweepCus) continue;
            ++chosen;
            std::set<std::tuple<int, int, int>> seen;
            int last = 0;
            for (int k = 0; k < all; ++k) {
                int r = k, g, n = 0;
                for (g = 0; g < t.most; ++g) {
                    n = 0;
                    for (int b = 0; b < B; ++b) n += groups[b] > g;
                    if (r < 2 * n) break;
                    r -= 2 * n;
                }
                int rank, slot, b = 0;
                place_of_ticket(r, n, 2, rank, slot);
                for (int before = 0; b < B; ++b) if (groups[b] > g && before++ == rank) break;
                if (g >= t.most || g < last || b >= B || slot < 0 || slot > 1) return fail("place", B, T, L, W, x);
                last = g;
                seen.insert({g, slot, b});
            }
            if ((int)seen.size() != all) return fail("two workgroups in one place", B, T, L, W, x);
        }
    }
    std::printf("%d offered, %d chosen\n", offered, chosen);
    return offered < 100 || chosen < 100;
}
"""


# What a launch takes, from the lengths alone: its table in float32 and in float64, and the groups of its longest sample.
CHOICE = r"""
#include <cstdio>
#include <vector>
#include "dag_chunks.h"
using namespace dagx;
int main() {
    static GroupTable tables[kMostTables];
    int B, T, L;
    while (std::scanf("%d %d %d", &B, &T, &L) == 3) {
        std::vector<int> len(B);
        for (int &n : len) if (std::scanf("%d", &n) != 1) return 1;
        for (int which = 0; which < 2; ++which) {
            TableChoice t;
            make_tables<1>(tables, t, B, T, L, L - 1, sweep_groups(B, L, L - 1), kMaxGroups, kSweepCosts, which);
            int used = 0;
            for (int x = t.ntable - 1; x > 0 && used == 0; --x) {
                int all = 0;
                for (const int n : len) all += 2 * (int)(t.ngroups[x] >> (4 * ((n >= 1 && n <= L ? (n + kBlk - 1) / kBlk : 1) - 1)) & 15);
                if (all <= kSweepCus) used = x;
            }
            std::printf("%d %d ", used, t.most);
        }
        std::printf("\n");
    }
}
"""


def _run(program, tmp_path, given=""):
    src, exe = tmp_path / "tables.hip", tmp_path / "tables"
    src.write_text(program)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-function",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "da_transformer_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, input=given)
    assert run.returncode == 0, run.stdout
    return run.stdout


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
def test_every_group_has_one_workgroup_whatever_table_is_chosen(tmp_path):
    _run(PROGRAM, tmp_path)


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
def test_the_batches_of_the_gpu_tests_take_the_tables_they_are_there_for(tmp_path):
    batches = [(B, T, L, table_lengths(B, L, T, shortest)[0].tolist()) for B, L, T, shortest, _, _ in TABLE_BATCHES]
    batches += [(len(ol), T, L, ol.tolist()) for T, L, ol in [mixed_lengths()]]
    given = "\n".join(" ".join(map(str, [B, T, L] + lengths)) for B, T, L, lengths in batches)
    got = [[int(n) for n in line.split()] for line in _run(CHOICE, tmp_path, given).splitlines()]
    assert [(x[0], x[2]) for x in got[:-1]] == [batch[5] for batch in TABLE_BATCHES]
    table32, most32, table64, most64 = got[-1]
    assert table32 > 0 and table64 > 0 and most32 != most64    # the two launches of a call lay the workspace out differently
