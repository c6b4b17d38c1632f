// The sweeps of dag_loss.hip (log-semiring) and dag_align.hip (max-semiring) in chunks of four steps: what a position block
// receives from the blocks below it is formed for four steps at once (in the loss on the matrix cores); only the 64 x 64
// triangle on the diagonal is walked step by step, by one wave.
#pragma once

#include <memory>

#include "dag_tiles.h"

namespace dagx {

// With SPACING 1 position block J works on chunk c (steps 4c+1 .. 4c+4) in stage J + c, with SPACING 2 in stage 2J + c; one
// barrier a stage is the only synchronisation of a workgroup.  What a block receives from the blocks below it is formed one
// stage ahead, by waves that are not on the critical path -- with SPACING 1 but for what it receives from block J - 1, which
// worked on that chunk only one stage earlier: that the walking wave itself forms when the stage begins.  So SPACING 1
// (the loss) has longer stages, by one tile, and one a block less: right where a tile is cheap beside a walk.
//
// In the loss numbers are linear: a cell holds exp(value - kap ln 2) 2^kShift with one integer exponent kap per block and step,
// chosen so that the block's largest cell lies in [2^(kShift-1), 2^kShift) -- in the float32 sweeps in every other step only,
// the others keep their scale (kSpare).  All scaling is by powers of two.
//
// The wide variant keeps cells, products and sums in float64; the staged transitions stay float32 registers (the register
// file holds no float64 tiles) and are converted as they are used.  What the float32 sweep cannot hold is, almost always,
// a cell far under the maximum of its block or a block far under its neighbours (inputs whose best prefixes are not the
// prefixes of the best paths); a float64 number has room for 1300 nats under its scale where a float32 number has 126.
constexpr int kChunk = 4;
constexpr int kDeadExp = -(1 << 30);        // the exponent of a block without a live cell
constexpr int kDeadBelow = -(1 << 29);      // any exponent below this is that of a dead block
constexpr int kMatchExpMax = 1 << 17;       // match values beyond 2^+-this are rounded (down: to this or 0; up: the sample is done again)
// In the float32 sweeps every other step does not scale its cells by their largest but lowers them by kSpare binades, which
// saves a reduction over the wave -- unless the largest has fallen below kScaleBelow, where the cells under it would lose
// range.  (Peaked samples of 700 nodes that the sweeps flagged: 41 of 128 without that exception, 29 with it; step by step
// sweeps flagged 65.  It costs 0.7 us of 106 at L = 512.)
constexpr int kSpare = 62;
constexpr float kScaleBelow = 4096.f;
constexpr int kChunkBlocks = 8;             // a group owns at most this many blocks: one wave walks one block

template <bool WIDE> struct Chunks;
template <> struct Chunks<false> {
    typedef float Cell;
    static constexpr int kShift = kShift2, kLinkShift = kShift2;   // powers of two that cells and staged transitions carry
    static constexpr int kFloor = -126;                            // least exponent of a scale factor in the upper sweep (0 below it in the lower)
    static constexpr int kStepPitch = 4;                           // distance of a cell's steps in a chunk of cells
};
template <> struct Chunks<true> {
    typedef double Cell;
    static constexpr int kShift = 850, kLinkShift = kShiftLinksWide;   // a sum of products: 2^(850 + 127 + 10) < 2^1024
    static constexpr int kFloor = -1022;
    static constexpr int kStepPitch = 2;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// Tiles that are multiplied out a stage ahead: those below the diagonal, with SPACING 1 but for the one next to it.
template <int SPACING>
__device__ __host__ __forceinline__ int tiles_of_block(int J, int W) { const int n = (J < W ? J : W) - (2 - SPACING); return n > 0 ? n : 0; }

// LDS of a group, in dwords.
struct ChunkLds {
    int depth;      // chunks of cells kept per block: read up to (blocks of the group) stages after they are written
    int runs;       // runs of tiles there can be
    int eb;         // [nsrc][depth][256]  cells of four steps, in the order of the products' first operand (cell_place)
    int kap;        // [nsrc][depth][4]    their exponents
    int part;       // [runs + 1][2][256]  products of a run of tiles (float32: four steps per lane; float64: [4][64]); behind them zeros
    int part_scale; // [nblk][2][4]        the exponents they are relative to
    int turn;       // float64: [nblk][256] where a walking wave turns the adjacent tile's product
    int frows, foff;// [nfor][256], [nfor][64]  landing areas of table rows and offsets of blocks of lower groups
    int both;       // [1]  counts the last two blocks' waves as they find their rows in memory
    int total;
};
__device__ __host__ inline ChunkLds chunk_lds(int jb0, int nblk, int W, bool wide) {
    ChunkLds o;
    const int flo = tile_ilo(jb0, W), nfor = jb0 - flo, nsrc = nfor + nblk, chunk = wide ? 512 : 256;
    int ntile = 0;
    for (int q = 0; q < nblk; ++q) ntile += tiles_of_block<1>(jb0 + q, W);
    const int reach = nblk < W ? nblk : W;
    o.depth = reach + 1 < 3 ? 3 : reach + 1;
    o.runs = ntile < kTileWaves + nblk - 1 ? ntile : kTileWaves + nblk - 1;
    int at = 0;
    o.eb = at; at += nsrc * o.depth * chunk;
    o.part = at; at += (o.runs + 1) * 2 * chunk;
    o.turn = at; at += wide ? nblk * chunk : 0;
    o.frows = at; at += nfor * 256;
    o.foff = at; at += nfor * 64;
    o.kap = at; at += nsrc * o.depth * 4;
    o.part_scale = at; at += nblk * 2 * 4;
    o.both = at; at += 4;
    o.total = at;
    return o;
}
// where a block's cell of step 4c + k, position `row`, stands in a chunk of cells: + kStepPitch k
template <bool WIDE>
__device__ __forceinline__ int cell_place(int row) {
    return WIDE ? ((row >> 3) * 16 + (row & 3) * 4) * 2 + ((row >> 2) & 1) : (row & 15) * 16 + (row >> 4);
}
constexpr int kForeign = 3;                  // foreign blocks a wave fetches at most
constexpr int kChunkLdsBytes = 160 * 1024 - 512;

// Those tiles, block by block, are dealt to the waves in runs: at most three to a wave that walks no block (a helper), at
// most SPACING to one that does (the triangle, and with SPACING 1 the tile next to it, take registers), and the foreign blocks
// to the helpers that fetch them: each to the wave that is done first with it.
struct TileDeal { unsigned wave; };          // four bits a wave: tiles, foreign blocks << 2
__device__ __host__ __forceinline__ int dealt_tiles(const TileDeal &d, int wave) { return (d.wave >> (4 * wave)) & 3; }
__device__ __host__ __forceinline__ int dealt_foreign(const TileDeal &d, int wave) { return (d.wave >> (4 * wave + 2)) & 3; }
// What a wave's pieces of a stage weigh in a plan: walking a block (with SPACING 1 with the product of the adjacent tile), a tile,
// fetching a foreign block (most of it waits); and how much of the sum of two waves' weights a SIMD takes for both, in per cent (waves w
// and w + 4 share one).  Set by timing calls, from the pieces' own times in hundreds of cycles on.
struct ChunkCosts { int walk, product, fetch, shared; };
// Returns how long the busiest wave or SIMD takes, -1 if there are more tiles than the waves have room for; alone: how long the busiest
// SIMD takes if it does nothing for one wave while it does something for the other.
template <int SPACING>
inline int deal_tiles(int jb0, int nblk, int W, const ChunkCosts &cost, TileDeal &deal, int &alone) {   // (on the host: a plan made by the kernel costs it 2 us)
    constexpr int kSimds = 4;
    int load[kTileWaves] = {0}, tiles[kTileWaves] = {0}, foreign[kTileWaves] = {0};
    for (int w = 0; w < nblk; ++w) load[w] = cost.walk - (SPACING == 1 && jb0 + w == 0 ? cost.product : 0);
    int ntile = 0;
    const int nfor = jb0 - tile_ilo(jb0, W);
    for (int q = 0; q < nblk; ++q) ntile += tiles_of_block<SPACING>(jb0 + q, W);
    auto busy = [&](const int w, const int more) {   // until when wave w (with `more` to do) keeps its SIMD or itself busy
        const int both = (load[w] + load[(w + kSimds) % kTileWaves] + more) * cost.shared / 100;
        return load[w] + more > both ? load[w] + more : both;
    };
    auto place = [&](int (&count)[kTileWaves], const bool fetch, const int work) {
        int best = -1, until = 0;
        for (int w = kTileWaves - 1; w >= 0; --w) {
            const int most = fetch ? (w >= nblk || nblk == kTileWaves ? kForeign : 0) : (w >= nblk ? kTilesPerWave : SPACING);
            if (count[w] >= most) continue;
            const int now = busy(w, work);
            if (best < 0 || now < until || (now == until && count[w] < count[best])) { best = w; until = now; }
        }
        if (best < 0) return false;
        ++count[best];
        load[best] += work;
        return true;
    };
    for (int n = 0; n < ntile; ++n) if (!place(tiles, false, cost.product)) return -1;
    for (int n = 0; n < nfor; ++n) if (!place(foreign, true, cost.fetch)) return -1;
    deal.wave = 0;
    int most = 0;
    alone = 0;
    for (int w = 0; w < kTileWaves; ++w) {
        deal.wave |= (unsigned)(tiles[w] | foreign[w] << 2) << (4 * w);
        most = busy(w, 0) > most ? busy(w, 0) : most;
        const int both = load[w] + load[(w + kSimds) % kTileWaves];
        alone = both > alone ? both : alone;
    }
    return most;
}
// first tile, number of tiles, first foreign block and number of foreign blocks of a wave (the helpers' tiles first,
// from the last wave down)
__device__ __host__ __forceinline__ void wave_tiles(const TileDeal &d, int wave, int &first, int &count) {
    first = 0; count = dealt_tiles(d, wave);
    for (int w = 1; w < kTileWaves; ++w) first += w > wave ? dealt_tiles(d, w) : 0;
}
__device__ __host__ __forceinline__ void wave_foreign(const TileDeal &d, int wave, int &first, int &count) {
    first = 0; count = dealt_foreign(d, wave);
    for (int w = 1; w < kTileWaves; ++w) first += w > wave ? dealt_foreign(d, w) : 0;
}

// Host: the groupings of a graph's position blocks for every number of blocks up to NB, each into at most C contiguous
// groups of at most kTileCap tiles (the diagonal ones among them) and kChunkBlocks blocks so that the busiest SIMD has
// least to do: as few groups as can be, or more even ones.  In a SIMD with a walk and little else the costs hide the other wave's work
// behind the walk; measured, a stage is longer by about a sixth of that, and by no more than the same share of the groups' mean.  So of
// the groupings with that bound the one whose busiest such SIMD has least is taken where that gains more than the further hand-overs
// take (one and a half stages each, of as many as a target of a fifth of the graph has).  us, as few as can be -> as measured with the
// groups here: alignment B = 1, L = 456, T = 182, transitions of at most 11 (two groups of four blocks -> four of two) 173.5 -> 159.5; B = 3,
// L = 811, T = 162, at most 166 (4 3 3 3 -> 3 2 2 2 2 2) 229 -> 216; B = 29, L = 240, T = 96, at most 27 94.6 -> 89.3; loss B = 58, L = 271,
// T = 54 (4 1 -> 3 2) 74.8 -> 69; and where as few as can be are kept: B = 12, L = 540, T = 67 120 against 124 with 3 2 1 1 1 1 for 4 2 1 1 1, B = 32,
// L = 452, T = 56, at most 92 89 against 93.  gtab[nb][g] .. gtab[nb][g+1]: blocks of group g (empty groups last).
template <int N>
struct ChunkPlan {
    // one of each for each set of costs
    unsigned char gtab[N][kMaxBlocksFast + 1][12];
    TileDeal deal[N][kMaxBlocksFast + 1][12];
    short busiest[N][kMaxBlocksFast + 1];         // how long the busiest SIMD of the graph's groups takes; kNoPlan: C groups do not hold it
};
constexpr int kNoPlan = 1 << 12;
// Every group there can be with a window, whatever the number of groups: group of blocks j .. j + n - 1.
template <int N>
struct GroupDeals {
    short cost[N][kMaxBlocksFast][kChunkBlocks + 1];   // -1: more tiles than a workgroup has room for
    TileDeal deal[N][kMaxBlocksFast][kChunkBlocks + 1];
    short alone[N][kMaxBlocksFast][kChunkBlocks + 1];
    short most[N], most_alone[N];                      // the greatest of them
    int spacing;
};
template <int SPACING, int N>
inline void deal_groups(int W, const ChunkCosts (&costs)[N], GroupDeals<N> &o) {
    o.spacing = SPACING;
    for (int x = 0; x < N; ++x) {
        o.most[x] = o.most_alone[x] = 0;
        for (int j = 0; j < kMaxBlocksFast; ++j) {
            int tiles = 0;
            for (int n = 1; n <= kChunkBlocks; ++n) {
                o.cost[x][j][n] = -1;
                o.deal[x][j][n] = TileDeal{0};
                if (j + n > kMaxBlocksFast) continue;
                tiles += j + n - tile_ilo(j + n - 1, W);
                int alone = 0;
                if (tiles <= kTileCap) o.cost[x][j][n] = (short)deal_tiles<SPACING>(j, n, W, costs[x], o.deal[x][j][n], alone);
                o.alone[x][j][n] = (short)alone;
                o.most[x] = o.cost[x][j][n] > o.most[x] ? o.cost[x][j][n] : o.most[x];
                o.most_alone[x] = o.alone[x][j][n] > o.most_alone[x] ? o.alone[x][j][n] : o.most_alone[x];
            }
        }
    }
}
template <int N>
inline void plan_chunks(const GroupDeals<N> &groups, int C, ChunkPlan<N> &plan) {
    for (int x = 0; x < N; ++x) {
        const auto &cost = groups.cost[x], &alone = groups.alone[x];
        for (int nb = 0; nb <= kMaxBlocksFast; ++nb) {
            int low = 0, high = groups.most[x] + 1;      // the least bound on a group's cost that C groups can keep
            unsigned char g[16];
            auto split = [&](const int most, const int most_alone) {   // (the second holds for groups that take `most`)
                int used = 0, j = 0;
                g[0] = 0;
                for (int q = 1; q < 16; ++q) g[q] = (unsigned char)nb;
                while (j < nb) {
                    int n = nb - j < kChunkBlocks ? nb - j : kChunkBlocks;
                    while (n > 0 && (cost[j][n] < 0 || cost[j][n] > most || (cost[j][n] == most && alone[j][n] > most_alone))) --n;
                    if (n == 0 || used == C) return false;
                    j += n;
                    g[++used] = (unsigned char)j;
                }
                return true;
            };
            // groups, how much longer than `high` the busiest SIMD of any takes if its waves' work does not overlap, and the sum over all
            auto over = [&](int &n, int &most, int &sum) {
                n = most = sum = 0;
                for (; n < C && g[n + 1] > g[n]; ++n) {
                    const int more = alone[g[n]][g[n + 1] - g[n]] - high;
                    most = more > most ? more : most;
                    sum += more > 0 ? more : 0;
                }
            };
            const int any = groups.most_alone[x];
            while (low < high) { const int mid = (low + high) / 2; if (split(mid, any)) high = mid; else low = mid + 1; }
            const bool ok = split(high, any);
            int n, most, sum;
            over(n, most, sum);
            if (ok && most > 0) {
                int n2, most2, sum2, low_alone = high, high_alone = high + most;
                while (low_alone < high_alone) { const int mid = (low_alone + high_alone) / 2; if (split(high, mid)) high_alone = mid; else low_alone = mid + 1; }
                split(high, high_alone);
                over(n2, most2, sum2);
                const long long stages = (16 + 5 * groups.spacing) * nb, cost = 90 * high * (n2 - n);   // (stages: five times)
                const bool pays = 2 * (most - most2) * stages > cost && 2 * (sum * n2 - sum2 * n) * stages > cost * n * n2;
                if (!pays) split(high, any);
            }
            plan.busiest[x][nb] = (short)(ok ? high : kNoPlan);
            for (int q = 0; q < 12; ++q) {
                plan.gtab[x][nb][q] = g[q];
                plan.deal[x][nb][q] = q < C && g[q + 1] > g[q] && g[q + 1] - g[q] <= kChunkBlocks ? groups.deal[x][g[q]][g[q + 1] - g[q]] : TileDeal{0};
            }
        }
    }
}
template <int SPACING, int N>
inline void plan_chunks(int W, int C, const ChunkCosts (&costs)[N], ChunkPlan<N> &plan) {
    GroupDeals<N> groups;
    deal_groups<SPACING>(W, costs, groups);
    plan_chunks(groups, C, plan);
}
// The deals and the plans for a window, remembered for the thread's later calls: C follows from the batch size, so that batches of
// changing size ask for several plans in turn, and the loss weighs the plans of several C in one call.  What these share, the deals of
// all groups, takes 10 to 20 us, a plan 3 to 10 (eleven plans with deals of their own 450 us, so 150).  At most kMaxBlocksFast windows'
// deals and kMaxBlocksFast * kMaxGroups plans, 1 to 2 KB each, given back when the thread ends.
inline int window_blocks(int translen) { const int w = (translen + kBlk - 1) / kBlk; return w < kMaxBlocksFast ? w : kMaxBlocksFast; }
template <int SPACING, int N>
inline const GroupDeals<N> &group_deals(int translen, const ChunkCosts (&costs)[N]) {
    static thread_local std::unique_ptr<GroupDeals<N>> deals[kMaxBlocksFast];
    const int W = window_blocks(translen);
    std::unique_ptr<GroupDeals<N>> &of = deals[W - 1];
    if (!of) {
        of.reset(new GroupDeals<N>);
        deal_groups<SPACING>(W, costs, *of);
    }
    return *of;
}
template <int SPACING, int N>
inline const ChunkPlan<N> &chunk_plan(int translen, int C, const ChunkCosts (&costs)[N]) {
    static thread_local std::unique_ptr<ChunkPlan<N>> plans[kMaxBlocksFast][kMaxGroups];
    std::unique_ptr<ChunkPlan<N>> &plan = plans[window_blocks(translen) - 1][C - 1];
    if (!plan) {
        plan.reset(new ChunkPlan<N>);
        plan_chunks(group_deals<SPACING>(translen, costs), C, *plan);
    }
    return *plan;
}

// ---- how many groups a sample gets (the loss) ----
// Table 0 has `least` groups for every sample, the others more for the longest samples and as many for shorter ones as it takes
// to keep the bound that the longest can keep: the time of a batch is that of its longest samples.  A launch takes the last
// table whose workgroups all find a CU; only the kernel knows the lengths, so it decides.  (B = 16, L = 1024, lengths from three
// quarters on: nine groups for samples of 16 blocks, six for 13, against eight for all: sweep, T = 256 330 -> 303 us, T = 128
// 213 -> 203; B = 14, L = 1000, T = 200 281 -> 257; B = 28, L = 640, T = 128 156 -> 147.)
struct GroupTable {
    unsigned char gtab[kMaxBlocksFast + 1][12];
    TileDeal deal[kMaxBlocksFast + 1][12];
};
constexpr int kMostTables = 3;
constexpr int kSweepCus = 256;          // workgroups of the sweeps that run side by side, one a CU
constexpr int kMostForTables = kWave;   // batches of at most this many samples choose: a lane looks at a sample's length
struct TableChoice {
    unsigned long long ngroups[kMostTables];   // (tables 1 ..) four bits for each number of blocks from 1 on: a sample's groups
    int ntable, least, most;                   // most: the most groups of any sample in any table
};
// Groups of a sample of nb blocks that keeps `bound` with as few as can be, at most c: the plan they are from and their number.
template <int SPACING, int N>
inline const ChunkPlan<N> &plan_for_bound(int translen, int c, int nb, int bound, const ChunkCosts (&costs)[N], int which, int &n) {
    int u = 1;
    while (u < c && chunk_plan<SPACING>(translen, u, costs).busiest[which][nb] > bound) ++u;
    const ChunkPlan<N> &plan = chunk_plan<SPACING>(translen, u, costs);
    for (n = 0; n < u && plan.gtab[which][nb][n + 1] > plan.gtab[which][nb][n];) ++n;
    return plan;
}
// Whether two sweeps of samples of seven eighths of L, with the bound that the longest keeps with c groups, would all find a CU.  (Where
// they would, most batches of ragged samples do; where all lengths are L and do not, the look at the lengths costs a few us: B = 20, L = 900,
// T = 180 332 -> 336, B = 17, L = 897 325 -> 328; of lengths from three quarters on 283 -> 230, from a third on 249 -> 227.)
template <int SPACING, int N>
inline bool typical_fits(int B, int L, int translen, int c, const ChunkCosts (&costs)[N], int which) {
    int n;
    plan_for_bound<SPACING>(translen, c, (7 * L / 8 + kBlk - 1) / kBlk, chunk_plan<SPACING>(translen, c, costs).busiest[which][(L + kBlk - 1) / kBlk], costs, which, n);
    return 2 * B * n <= kSweepCus;
}
inline bool may_choose(int B, int L) { return B <= kMostForTables && L > 4 * kBlk; }
// A table is offered where the longest sample's stages (one a chunk, one a block, one and a half a hand-over) take at most 97 %
// of what they take in `least` groups and are shorter by a twelfth of a walk (with a bound of 48 already, groups for one of 45, a
// walk alone, lose: B = 32, L = 512, T = 256 216 -> 227 us, T = 170 158 -> 165; B = 13, L = 458, T = 157 143.5 -> 149), and
// where two sweeps of samples of seven eighths of L would all find a CU.  room: the most groups a sweep that the caller's workspace has
// pipeline words for; with `least` there is only table 0.
template <int SPACING, int N>
inline void make_tables(GroupTable (&tables)[kMostTables], TableChoice &o, int B, int T, int L, int translen, int least, int room,
                        const ChunkCosts (&costs)[N], int which) {
    auto plan_of = [&](const int c) -> const ChunkPlan<N> & { return chunk_plan<SPACING>(translen, c, costs); };
    auto copy_row = [&](GroupTable &table, const int nb, const ChunkPlan<N> &plan) {
        for (int q = 0; q < 12; ++q) { table.gtab[nb][q] = plan.gtab[which][nb][q]; table.deal[nb][q] = plan.deal[which][nb][q]; }
    };
    o.ntable = 1;
    o.least = o.most = least;
    const int NB = (L + kBlk - 1) / kBlk, NC = (T - 1 + kChunk - 1) / kChunk;
    for (int nb = 0; nb <= kMaxBlocksFast; ++nb) copy_row(tables[0], nb, plan_of(least));
    if (!may_choose(B, L) || room <= least) return;
    auto stages2 = [&](const int c) { return 2 * (NC + NB) + 3 * (c - 1); };
    const int first = plan_of(least).busiest[which][NB];
    int best = first;
    const long long now = (long long)first * stages2(least);
    for (int c = least + 1; c <= kMaxGroups && c <= NB && o.ntable < kMostTables; ++c) {
        const int bound = plan_of(c).busiest[which][NB];
        if (bound >= best || 12 * (first - bound) < costs[which].walk || 100 * (long long)bound * stages2(c) > 97 * now) continue;
        GroupTable &table = tables[o.ntable];
        unsigned long long ngroups = 0;
        int most = 1;
        if (!typical_fits<SPACING>(B, L, translen, c, costs, which)) continue;
        for (int nb = 0; nb <= kMaxBlocksFast; ++nb) {
            if (nb < 1 || nb > NB) { copy_row(table, nb, plan_of(c)); continue; }
            int n;
            copy_row(table, nb, plan_for_bound<SPACING>(translen, c, nb, bound, costs, which, n));
            ngroups |= (unsigned long long)n << (4 * (nb - 1));
            most = n > most ? n : most;
        }
        if (most > room) continue;
        o.ngroups[o.ntable++] = ngroups;
        o.most = most > o.most ? most : o.most;
        best = bound;
    }
}
// Ticket r among those of the n samples that have a certain group -> which of the samples, which of its sweeps: a sample's
// two sweeps eight tickets apart while there are eight samples more (so they mostly share an XCD).
__device__ __host__ __forceinline__ void place_of_ticket(int r, int n, int ndir, int &rank, int &slot) {
    const int full = n & ~7, rest = n - full > 0 ? n - full : 1;
    if (r < ndir * full) { rank = (r / (8 * ndir)) * 8 + r % 8; slot = (r / 8) % ndir; }
    else { r -= ndir * full; rank = full + r % rest; slot = r / rest; }
}

// Workgroups per sweep (two sweeps a sample) in table 0: as few as hold the tiles, but with at most four blocks each, one walk to a
// SIMD, where the device has a CU for every workgroup (with the plans before there were tables, forward, up to eight -> up to four
// blocks: B = 40, L = 328, T = 41 67 -> 61 us; B = 16, L = 512, T = 64 102 -> 97.5; B = 64 and transitions of at most 32 88 -> 79; B = 16,
// L = 1024 and transitions of at most 64 122 -> 104).  Where a table may have more groups the two come out the same now (62.6 and 62.1;
// 89.6 and 90.2; 82.7 and 82.2; T = 128 144.8 and 144.4): the line decides for workspaces that have room for table 0 alone.
inline int sweep_groups(int B, int L, int translen) {
    const int C = groups_needed(L, translen, 4), sweeps = 2 * ((B + 7) & ~7);
    return (long long)sweeps * C <= kSweepCus && C > 0 ? C : groups_needed(L, translen, kChunkBlocks);
}
// float32, float64.  Found by timing the sweeps themselves under some forty sets (us; first the costs of each piece timed alone,
// with a SIMD taking the sum of its two waves' work, {45, 7, 4, 100} and {85, 17, 11, 100}; then these): float32 B = 64, L = 512, T = 64
// 107 -> 95; B = 16, L = 1024, T = 256 347 -> 329; B = 16, L = 512, T = 128 134 -> 127; B = 8, L = 1024, T = 256 334 -> 302; float64 at the
// first of them 151 -> 141.  A fetched block waits for the rows of its producer and for LDS twice, so it keeps its wave for longer than
// its instructions take; and while a wave waits, the other wave of its SIMD works.
constexpr ChunkCosts kSweepCosts[2] = {{45, 9, 12, 70}, {85, 25, 16, 80}};

// ---- the alignment's rules ----
// Whether the sweep goes in chunks of four steps.  They cost T / 4 stages and one or two more for every block of nodes, single
// steps T of two fifths of that, and a stage of four steps is hardly longer where the sums are formed by matrix instructions: even
// at about two steps for every block and 22 more, where windows are short and a step has few tiles at four and 14 (alignment, steps
// and chunks, us: B = 64, L = 512, T = 28 76.9 and 75.2, T = 40 98.4 and 87.3; B = 16, L = 768, T = 36 110 and 108, T = 48 135 and 124; B = 64, L = 640,
// T = 40 112 and 109; B = 1, L = 900, T = 52 150 and 152, T = 60 165 and 162; B = 40, L = 1024, T = 56 227 and 187; B = 64, L = 320, T = 32
// 55.7 and 55.6; B = 200, L = 256, T = 30 54.6 and 55.9; transitions of at most 100: B = 16, L = 768, T = 60 108 and 110; B = 1, L = 900, T = 75 135 and 128).
// Eight blocks of a workgroup each, with two stages a block, take longest to fill: 43 (L = 512: B = 1, T = 40 76.7 and 79.7; B = 16, T = 40 83.2 and
// 86.3, T = 48 87.9 and 87.7; B = 32, T = 38 83.5 and 87.5, T = 44 89.1 and 88.4).  Up to three blocks the line is at six for every block and 8 more.
// (The line is that of few samples.  With more it could be lower for most sizes, but not for all: B = 64, L = 256, T = 26 44.7 and 44.5, B = 200
// 50.5 and 53.5; L = 1024, T = 32 B = 40 155 and 148, B = 1 114 and 133.)
inline bool align_in_chunks(int B, int T, int L, int translen) {
    const int NB = (L + kBlk - 1) / kBlk, most = 6 * NB + 8;
    const int line = window_blocks(translen) <= 3 ? 4 * NB + 14 : NB == 8 && ((B + 7) & ~7) * NB <= 256 ? 43 : 2 * NB + 22;
    return T >= (line < most ? line : most) && (int64_t)B * L * translen >= 4;   // (the chunked kernel's tiles are loaded four elements at a time)
}

// Workgroups per sweep.  In chunks: from four position blocks on as many as the device has room for (one per CU) up to one
// for each block, at most ten.  (Fewer tiles a SIMD, against more hand-overs: as many as hold the tiles -> this, alignment of
// B = 16, L = 1024, T = 256 504 -> 423 us; B = 16, L = 768, T = 192 365 -> 267; B = 4, L = 700, T = 110 250 -> 178; B = 64, L = 320,
// T = 48 90 -> 72; B = 64, L = 256, T = 64 91 -> 75.)  Step by step: twice as many as hold the tiles where there is room and the graph has at least four
// blocks (5 to 13 %; more lose); where that exceeds what the kernel supports, ten when they fit.
inline int align_groups(int B, int T, int L, int translen) {
    const int NB = (L + kBlk - 1) / kBlk, B8 = (B + 7) & ~7;
    if (align_in_chunks(B, T, L, translen)) {
        const int C = groups_needed(L, translen, kChunkBlocks);
        if (C == 0 || NB < 4) return C;
        const int room = 256 / B8, most = NB < 10 ? NB : 10, more = room < most ? room : most;
        return more > C ? more : C;
    }
    const int C = groups_needed(L, translen, kMaxBlocksFast);
    if (C == 0) return 0;
    if (NB >= 4 && 2 * C <= kMaxGroups && 2 * C <= NB && (long long)B8 * 2 * C <= 256) return 2 * C;
    return C < 10 && NB >= 10 && (long long)B8 * 10 <= 256 ? 10 : C;
}
// Stages from a block's walk of a chunk to the next block's: see dag_align_chunks_kernel.
inline int align_spacing(int NB, int C) { return NB <= 5 || (NB <= 8 && 2 * NB <= 3 * C) ? 2 : 1; }
// The alignment's weights: those that timing calls under some twenty sets found when its sums were formed by vector instructions.  A tile
// takes half as long now and two waves of a SIMD hardly less than one after the other, but some ten sets timed again found none better, and
// weights by the pieces' times of today, {45 or 30, 13, 4, 100}, are worse: alignment, us, these and those, B = 64, L = 512, T = 64 101.6 and 104,
// B = 16, L = 768, T = 192 230 and 238, B = 4, L = 700, T = 110 151 and 159, B = 64, L = 256, T = 64 (SPACING 2) 65.0 and 68.4, B = 40, L = 400,
// T = 60 (SPACING 2) 88.5 and 93.2.  With SPACING 1 a fetched block weighs 2 where windows span more than three blocks, so that a group
// fetches many and their waits overlap, else 4.  With 4 for all: B = 9, L = 876, T = 175 254 us for 250, B = 2, L = 846, T = 338 369 for 364
// (but B = 41, L = 944, T = 283 418 for 429); with 2 for all: B = 91, L = 896, T = 358, transitions of at most 65 481 for 467, B = 74, L = 468, T = 58,
// at most 139 92.0 for 88.6, B = 14, L = 955, T = 238, at most 113 269 for 246.
template <int SPACING>
constexpr ChunkCosts kAlignCosts[2][1] = {{SPACING == 1 ? ChunkCosts{62, 27, 2, 65} : ChunkCosts{36, 27, 4, 55}},
                                          {SPACING == 1 ? ChunkCosts{62, 27, 4, 65} : ChunkCosts{36, 27, 4, 55}}};
template <int SPACING>
inline const ChunkCosts (&align_costs(int translen))[1] { return kAlignCosts<SPACING>[window_blocks(translen) <= 3]; }

// LDS of a group, in dwords: cells of four steps in the order of the table, results of a wave's tiles that lead to one block.
struct AlignLds {
    int depth, runs;    // chunks of cells kept per block; runs of tiles there can be
    int eb;             // [nsrc][depth][4][64]
    int both;           // [1] SPACING 1: counts the last two blocks' waves as they find their rows in memory
    int part, from;     // [runs][2][64][4] best scores of four steps a lane; [runs][2][64] the blocks they come from, a byte each
    int total;
};
__device__ __host__ inline AlignLds align_lds(int jb0, int nblk, int W, int spacing) {
    AlignLds o;
    const int nsrc = jb0 - tile_ilo(jb0, W) + nblk;
    int ntile = 0;
    for (int q = 0; q < nblk; ++q) ntile += spacing == 1 ? tiles_of_block<1>(jb0 + q, W) : tiles_of_block<2>(jb0 + q, W);
    // (read up to SPACING (blocks of the group) stages after they are written; foreign rows are copied into place up to a
    // stage before they are due)
    o.depth = spacing * (nblk < W ? nblk : W) + 3 - spacing;
    o.runs = ntile < kTileWaves + nblk - 1 ? ntile : kTileWaves + nblk - 1;
    int at = 0;
    o.eb = at; at += nsrc * o.depth * 256;
    o.part = at; at += o.runs * 2 * 256;
    o.from = at; at += o.runs * 2 * 64;
    o.both = at; at += 4;
    o.total = at;
    return o;
}

// ---- what a wave has to do, worked out at the start of the kernel ----
// A run is a wave's tiles that lead to one block; runs are numbered in the order of the tiles.
struct WaveTiles {
    int count;                                     // tiles to multiply out a stage ahead
    int I[kTilesPerWave], q[kTilesPerWave];        // source block, own block it leads to (a walking wave: slot 2 the triangle, with
                                                   // SPACING 1 slot 0 the tile next to it)
    int run[kTilesPerWave];                        // run it belongs to
    bool ok[kTilesPerWave], start[kTilesPerWave], end[kTilesPerWave], lead[kTilesPerWave];   // (slots to multiply out a stage ahead;) first / last tile of its run; run that begins with the block's first tile
    bool adjacent;                                 // slot 0 holds a tile next to the diagonal
    int run_first, run_count;                      // the runs that lead to the block this wave walks
};
template <int SPACING>
__device__ __forceinline__ WaveTiles plan_wave(const TileDeal &deal, int jb0, int nblk, int W, int none, int wave, int lane) {
    WaveTiles t;
    const int flo = tile_ilo(jb0, W);
    const bool owner = wave < nblk;
    int my_first;
    wave_tiles(deal, wave, my_first, t.count);
    // lane <-> block (f: its first tile) and lane <-> wave (w_first: its first tile)
    int f = 0, w_first, w_count;
#pragma unroll
    for (int q = 0; q < kChunkBlocks; ++q) f += q < lane && q < nblk ? tiles_of_block<SPACING>(jb0 + q, W) : 0;
    wave_tiles(deal, lane & (kTileWaves - 1), w_first, w_count);
    int f_of[kChunkBlocks + 1];
    bool cuts = lane < kTileWaves && w_count > 0;   // this wave's first tile begins a run in the middle of a block
#pragma unroll
    for (int q = 0; q <= kChunkBlocks; ++q) {
        f_of[q] = __builtin_amdgcn_readlane(f, q);
        if (q < nblk) cuts = cuts && !(w_first == f_of[q] && tiles_of_block<SPACING>(jb0 + q, W) > 0);
    }
    const int without = jb0 < 3 - SPACING ? 3 - SPACING - jb0 : 0;   // (block 0, with SPACING 1 also block 1, has no such tiles)
    // number of runs that begin at or before tile n of block q
    auto runs_to = [&](const int q, const int n) { return q + 1 - without + (int)__builtin_popcountll(__builtin_amdgcn_ballot_w64(cuts && w_first <= n)); };
#pragma unroll
    for (int u = 0; u < kTilesPerWave; ++u) {
        const int r0 = SPACING == 1 && owner ? u - 1 : u, n = my_first + r0;
        t.ok[u] = r0 >= 0 && r0 < t.count;
        int q = 0;
#pragma unroll
        for (int x = 1; x < kChunkBlocks; ++x) q = x < nblk && n >= f_of[x] ? x : q;
        const int lo = tile_ilo(jb0 + q, W), r = n - f_of[q];
        t.q[u] = t.ok[u] ? q : 0;
        t.I[u] = t.ok[u] ? lo + r : flo;
        t.start[u] = r0 == 0 || r == 0;
        t.end[u] = r0 == t.count - 1 || lo + r == jb0 + q - (3 - SPACING);
        t.lead[u] = r0 >= r;
        t.run[u] = runs_to(q, n) - 1;
    }
    t.run_first = none; t.run_count = 1;           // (a block without such tiles)
    if (owner && tiles_of_block<SPACING>(jb0 + wave, W) > 0) {
        const int n = __builtin_amdgcn_readlane(f, wave);
        t.run_first = runs_to(wave, n) - 1;
        t.run_count = runs_to(wave, n + tiles_of_block<SPACING>(jb0 + wave, W) - 1) - t.run_first;
    }
    t.adjacent = SPACING == 1 && owner && jb0 + wave > 0;
    if (owner) {
        t.I[kTilesPerWave - 1] = jb0 + wave; t.q[kTilesPerWave - 1] = wave;
        if (SPACING == 1) { t.I[0] = jb0 + wave - (t.adjacent ? 1 : 0); t.q[0] = wave; }
    }
    return t;
}

// a = {a's lower half, b's lower half}, b = {a's upper half, b's upper half}.  (The results go through unsigned variables:
// __builtin_bit_cast of an element of a vector yields element 0 with this compiler.)
__device__ __forceinline__ void swap_halves(float &a, float &b) {
    const u32x2 s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    const unsigned x = s[0], y = s[1];
    a = __builtin_bit_cast(float, x); b = __builtin_bit_cast(float, y);
}

// the largest of 64 numbers >= 0 as its bits, wave-uniform (a NaN is passed over)
__device__ __forceinline__ unsigned wave64_max_positive(float x) {
    unsigned v = __builtin_bit_cast(unsigned, x);
    asm("s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
        : "+v"(v));
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
// the largest of 64 integers, wave-uniform
__device__ __forceinline__ int wave64_max_int(int v) {
    asm("s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
        : "+v"(v));
    return __builtin_amdgcn_readlane(v, 63);
}
// {largest x, largest y} over the 64 lanes: lanes 0..31 of the result are to be reduced for x, 32..63 for y
__device__ __forceinline__ float fold_two(float x, float y) { swap_halves(x, y); return __builtin_fmaxf(x, y); }
// four maxima over the 64 lanes, each in lane 63 (side by side: no wait states between dependent steps); PAIR: beside them those
// over either half of a fifth, in lanes 31 and 63
template <bool PAIR>
__device__ __forceinline__ void wave64_max4(float (&v)[4], float &pair) {
    if constexpr (PAIR)
        asm("s_nop 1\n\t"
            "v_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %4, %4, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %4, %4, %4 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %4, %4, %4 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %4, %4, %4 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %4, %4, %4 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_bcast:31 row_mask:0xc bank_mask:0xf"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(pair));
    else
        asm("s_nop 1\n\t"
            "v_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_max_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "v_max_f32_dpp %1, %1, %1 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "v_max_f32_dpp %2, %2, %2 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "v_max_f32_dpp %3, %3, %3 row_bcast:31 row_mask:0xc bank_mask:0xf"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}
// ... those over either half alone
__device__ __forceinline__ void half_max(float &pair) {
    asm("s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf"
        : "+v"(pair));
}
// max over the lanes with the same lane & 3, in every lane
__device__ __forceinline__ int by_step_max(int v) {
    asm("s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(v));
    u32x2 p = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    v = max((int)p[0], (int)p[1]);
    p = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return max((int)p[0], (int)p[1]);
}

// max over the sixteen lanes of a row, in every lane
__device__ __forceinline__ int row16_max_int(int v) {
    asm("s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_i32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf"
        : "+v"(v));
    return v;
}

// g[t] += f[lane t of the row] * a[t]: four steps, each with its own factor
__device__ __forceinline__ void scaled4(f32x4 &g, float f, f32x4 a) {
    float g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf"
        : "+v"(g0), "+v"(g1), "+v"(g2), "+v"(g3) : "v"(f), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]));
    g = f32x4{g0, g1, g2, g3};
}

// sum over the 64 rows of a tile for four steps: out[t] = sum_k e[k][t] P[k][lane].  e[q] holds rows 16q .. 16q+15,
// lane 4 (k & 15) + t.  v_mfma_f32_4x4x1_16b multiplies, per 4-lane block, a 4 x 1 by a 1 x 4; with the first operand of
// block abid broadcast to all sixteen (cbsz 4) that is four steps times 64 positions of one row.  Two chains of
// accumulators: a dependent one issues every 12 cycles, two every 9.
__device__ __forceinline__ f32x4 tile_product(const Tile &t, f32x4 e) {
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#define DAGX_PAIR(q, k) \
    x = __builtin_amdgcn_mfma_f32_4x4x1f32(e[q], t.p[16 * (q) + (k)], x, 4, (k), 0); \
    y = __builtin_amdgcn_mfma_f32_4x4x1f32(e[q], t.p[16 * (q) + (k) + 1], y, 4, (k) + 1, 0);
#define DAGX_ROWS(q) DAGX_PAIR(q, 0) DAGX_PAIR(q, 2) DAGX_PAIR(q, 4) DAGX_PAIR(q, 6) DAGX_PAIR(q, 8) DAGX_PAIR(q, 10) DAGX_PAIR(q, 12) DAGX_PAIR(q, 14)
    DAGX_ROWS(0) DAGX_ROWS(1) DAGX_ROWS(2) DAGX_ROWS(3)
#undef DAGX_ROWS
#undef DAGX_PAIR
    return x + y;
}

// The same in float64, four steps times sixteen positions per accumulator: out[g], lane 16 m + o: step m, position 16 g + o.
// v_mfma_f64_4x4x4_4b: first operand lane 4 b + m + 16 k = step m of row k (the same in all four blocks b), second lane
// 4 b + n + 16 k = row k, position 4 b + n, result lane 4 b + 16 m + n.  Tile register 16 g + j: row 4 j + lane / 16,
// position 16 g + lane mod 16.  (A float64 product takes 16.5 cycles, its operand's conversion 4 to 5.)
__device__ __forceinline__ void tile_product(const Tile &t, const double *cells, int lane, double (&out)[4]) {
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    const f64x2 *const e = reinterpret_cast<const f64x2 *>(cells) + (lane >> 4) * 4 + (lane & 3);
#pragma unroll
    for (int g = 0; g < 4; ++g) out[g] = 0.0;
#pragma unroll
    for (int jp = 0; jp < 8; ++jp) {
        const f64x2 ev = e[16 * jp];
        const double e0 = ev[0], e1 = ev[1];
        // (by hand: the compiler would convert ahead of the loop over the stages, for which there are no registers.  A product
        // reads its operands two wait states after a vector instruction has written them.)
        double b[8];
        asm volatile("v_cvt_f64_f32 %0, %8\n\t"
                     "v_cvt_f64_f32 %1, %9\n\t"
                     "v_cvt_f64_f32 %2, %10\n\t"
                     "v_cvt_f64_f32 %3, %11\n\t"
                     "v_cvt_f64_f32 %4, %12\n\t"
                     "v_cvt_f64_f32 %5, %13\n\t"
                     "v_cvt_f64_f32 %6, %14\n\t"
                     "v_cvt_f64_f32 %7, %15\n\t"
                     "s_nop 1"
                     : "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3]), "=&v"(b[4]), "=&v"(b[5]), "=&v"(b[6]), "=&v"(b[7])
                     : "v"(t.p[2 * jp]), "v"(t.p[16 + 2 * jp]), "v"(t.p[32 + 2 * jp]), "v"(t.p[48 + 2 * jp]),
                       "v"(t.p[2 * jp + 1]), "v"(t.p[16 + 2 * jp + 1]), "v"(t.p[32 + 2 * jp + 1]), "v"(t.p[48 + 2 * jp + 1]));
#pragma unroll
        for (int g = 0; g < 4; ++g) out[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(e0, b[g], out[g], 0, 0, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) out[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(e1, b[4 + g], out[g], 0, 0, 0);
    }
}

// The triangle on the diagonal (row i of a tile reaches lanes j > i only) in 48 registers instead of 64:
//   p[0..31]:  lanes 0..31 rows 0..31, lanes 32..63 rows 32..63 -- the two 32 x 32 triangles side by side;
//   p[32..47]: the square between them, lanes 32..63 rows 0..15, lanes 0..31 rows 16..31 of positions lane + 32.
__device__ __forceinline__ void fold_triangle(Tile &t, int lane) {
    const bool hi = lane >= 32;
    float sq[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        float x = t.p[16 + k], y = t.p[k];
        swap_halves(x, y);       // y: lanes 0..31 have row 16 + k of lane + 32, lanes 32..63 row k
        sq[k] = y;
    }
#pragma unroll
    for (int r = 0; r < 32; ++r) t.p[r] = hi ? t.p[32 + r] : t.p[r];
#pragma unroll
    for (int k = 0; k < 16; ++k) t.p[32 + k] = sq[k];
}
// sum_i e[i] P[i][lane] over the folded triangle; upper_half: 0 in lanes 0..31, 1 in lanes 32..63.
// v_permlane16_swap makes the rows {0,0,2,2} and {1,1,3,3} of e, v_permlane32_swap the rows {1,1,0,0} of those, another
// one adds up the two halves' shares of the square.  A lane swap and a DPP operand want their source two wait states
// old: the moves and swaps stand among the FMAs so that only the first needs an s_nop (one costs as much as two FMAs).
__device__ __forceinline__ float triangle_dot(const Tile &t, float e, float upper_half) {
    float a, b, b2, odd, crossed, rest;
    asm("v_mov_b32 %2, %1\n\t"
        "s_nop 1\n\t"
        "v_permlane16_swap_b32 %1, %2\n\t"
        "v_mov_b32 %3, %2\n\t"
        "v_mov_b32 %4, %1\n\t"
        "v_mul_f32_dpp %0, %1, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_permlane32_swap_b32 %3, %4\n\t"
        "v_fmac_f32_dpp %0, %1, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %18 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %19 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %20 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "=&v"(a), "+v"(e), "=&v"(odd), "=&v"(crossed), "=&v"(rest)
        : "v"(t.p[0]), "v"(t.p[1]), "v"(t.p[2]), "v"(t.p[3]), "v"(t.p[4]), "v"(t.p[5]), "v"(t.p[6]), "v"(t.p[7]), "v"(t.p[8]), "v"(t.p[9]), "v"(t.p[10]), "v"(t.p[11]), "v"(t.p[12]), "v"(t.p[13]), "v"(t.p[14]), "v"(t.p[15]));
    asm("v_mul_f32_dpp %0, %1, %2 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %3 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %4 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %5 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %6 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %7 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %8 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %9 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %10 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %11 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %12 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %13 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %14 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %15 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %16 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %17 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "=&v"(b) : "v"(crossed), "v"(t.p[32]), "v"(t.p[33]), "v"(t.p[34]), "v"(t.p[35]), "v"(t.p[36]), "v"(t.p[37]), "v"(t.p[38]), "v"(t.p[39]), "v"(t.p[40]), "v"(t.p[41]), "v"(t.p[42]), "v"(t.p[43]), "v"(t.p[44]), "v"(t.p[45]), "v"(t.p[46]), "v"(t.p[47]));
    asm("v_mov_b32 %2, %1\n\t"
        "v_fmac_f32_dpp %0, %3, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_permlane32_swap_b32 %1, %2\n\t"
        "v_fmac_f32_dpp %0, %3, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %18 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %19 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %3, %20 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32 %1, %1, %2\n\t"
        "v_fmac_f32 %0, %1, %4"
        : "+v"(a), "+v"(b), "=&v"(b2) : "v"(odd), "v"(upper_half), "v"(t.p[16]), "v"(t.p[17]), "v"(t.p[18]), "v"(t.p[19]), "v"(t.p[20]), "v"(t.p[21]), "v"(t.p[22]), "v"(t.p[23]), "v"(t.p[24]), "v"(t.p[25]), "v"(t.p[26]), "v"(t.p[27]), "v"(t.p[28]), "v"(t.p[29]), "v"(t.p[30]), "v"(t.p[31]));
    return a;
}

// the same in float64: each row is converted as it is used
__device__ __forceinline__ void fma16_rowbcast(double &acc, double e, const float *p) {
    double t0, t1;
    asm("s_nop 1\n\t"
        "v_cvt_f64_f32 %1, %4\n\t"
        "v_cvt_f64_f32 %2, %5\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %6\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %7\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %8\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %9\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %10\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %11\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %12\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %13\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %14\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %15\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %16\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %17\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %1, %18\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f64_f32 %2, %19\n\t"
        "v_fmac_f64_dpp %0, %3, %1 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_fmac_f64_dpp %0, %3, %2 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "+v"(acc), "=&v"(t0), "=&v"(t1)
        : "v"(e), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]),
          "v"(p[8]), "v"(p[9]), "v"(p[10]), "v"(p[11]), "v"(p[12]), "v"(p[13]), "v"(p[14]), "v"(p[15]));
}
// {x, y} -> x: rows {x0 y0 x2 y2} / halves {x.lo, y.lo}; y: rows {x1 y1 x3 y3} / halves {x.hi, y.hi}
template <int LANES>
__device__ __forceinline__ void swap_lanes(double &x, double &y) {
    const unsigned long long xb = __builtin_bit_cast(unsigned long long, x), yb = __builtin_bit_cast(unsigned long long, y);
    unsigned word[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const unsigned xw = (unsigned)(xb >> (32 * h)), yw = (unsigned)(yb >> (32 * h));
        const u32x2 s = LANES == 16 ? __builtin_amdgcn_permlane16_swap(xw, yw, false, false) : __builtin_amdgcn_permlane32_swap(xw, yw, false, false);
        word[0][h] = s[0]; word[1][h] = s[1];
    }
    x = __builtin_bit_cast(double, (unsigned long long)word[0][1] << 32 | word[0][0]);
    y = __builtin_bit_cast(double, (unsigned long long)word[1][1] << 32 | word[1][0]);
}
__device__ __forceinline__ double triangle_dot(const Tile &t, double e, float upper_half) {
    double even = e, odd = e;
    swap_lanes<16>(even, odd);                 // rows {0,0,2,2} and {1,1,3,3} of e
    double crossed = odd, rest = even;
    swap_lanes<32>(crossed, rest);             // rows {1,1,0,0}
    double a = 0.0, b = 0.0;
    fma16_rowbcast(a, even, t.p);
    fma16_rowbcast(b, crossed, t.p + 32);
    fma16_rowbcast(a, odd, t.p + 16);
    double other = b;
    swap_lanes<32>(b, other);
    return a + (b + other) * (double)upper_half;
}

// ---- staging -----------------------------------------------------------------------------------------------------
// A tile's 64 x 64 transitions, loaded four neighbouring elements a lane (sixteen lanes a row), converted, and turned
// through LDS into lane <-> output position.  What bounds staging is the number of vector-memory instructions: a CU
// takes one per 26 cycles whatever its width, so 64 loads of one element each cost a tile of a full workgroup
// 12 000 cycles, and the kernel 15 us at L = 512.
//   alpha: row n of the patch is predecessor 64 I + n, memory runs along the output positions;
//   beta:  row n is output position 64 J + n (node L_b - 1 - 64 J - n), memory runs against the predecessors.
// The patch holds them as [row][column]: columns ascending with memory, so 63 - (position in block I) for beta.
constexpr int kPatchPitch = kBlk + 4;      // (16-byte rows; 64 lanes a row apart meet every bank alike)
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
template <typename TL> struct Quad;
template <> struct Quad<float> { typedef f32x4 V; __device__ __forceinline__ static float get(V v, int k) { return v[k]; } };
template <> struct Quad<__half> { typedef h16x4 V; __device__ __forceinline__ static float get(V v, int k) { return (float)v[k]; } };
template <> struct Quad<bf16_t> { typedef u16x4 V; __device__ __forceinline__ static float get(V v, int k) { return __uint_as_float((unsigned)v[k] << 16); } };

// one tile -> exp(E) 2^SHIFT (or E itself: !EXP) in the wave's patch; `tiny` as in link_prob.  before / behind: how many elements the
// tensor has in front of and behind the sample, where a load may reach (into places that are masked).
template <typename TL, int SHIFT, bool EXP = true, int BATCH = 16>
__device__ __forceinline__ void stage_tile(float *patch, const TL *links, int I, int J, int lane, int dir, int Lb, int translen, int last_index,
                                           int before, int behind, float tiny) {
    typedef typename Quad<TL>::V V;
    const int dd = (J - I) * kBlk - 1, n0 = lane >> 4, c = 4 * (lane & 15);
    const int index0 = dir == 0 ? (I * kBlk + n0) * translen + dd + c - n0 : (Lb - 1 - J * kBlk - n0) * translen + dd + n0 - c - 3;
    const int step = 4 * (dir == 0 ? translen - 1 : 1 - translen);
    const int lowest_i = min(index0, index0 + 15 * step), highest_i = max(index0, index0 + 15 * step) + 3;
    float *const dst = patch + n0 * kPatchPitch + (dir == 0 ? c : kBlk - 4 - c);
    // element k of group g (row n0 + 4 g): its distance is d0 + g dstep + k; it has a place in the sample for k < k_end(g0 + g)
    const int d0 = dir == 0 ? dd + c - n0 : dd + n0 - c - 3, dstep = dir == 0 ? -4 : 4;
    auto k_end = [&](const int g) { return dir == 0 ? Lb - J * kBlk - c : (J * kBlk + n0 + 4 * g < Lb ? 4 : 0); };
    auto valid = [&](const int g, const int k, const int ke) { return (unsigned)(d0 + g * dstep + k) < (unsigned)translen && k < ke; };
    const int back = kBlk * translen + 4 * kBlk;   // (an unsigned offset from a scalar base: one register a load)
    const char *const base = reinterpret_cast<const char *>(links) - (int64_t)back * (int64_t)sizeof(TL);
    auto load = [&](const int at) { V v; __builtin_memcpy(&v, base + (unsigned)(at + back) * (unsigned)sizeof(TL), sizeof(V)); return v; };
    // every (row, column) of the tile is a transition of the sample
    const bool interior = J > I && dd + kBlk - 1 < translen && J * kBlk + kBlk - 1 < Lb;
    const bool inside = __builtin_amdgcn_ballot_w64(lowest_i < -before || highest_i > last_index + behind) == 0;
    // (BATCH loads in flight: sixteen, fewer where the registers would not do)
#pragma unroll
    for (int g0 = 0; g0 < 16; g0 += BATCH) {
        if (BATCH < 16) __builtin_amdgcn_sched_barrier(0);
        V raw[BATCH];
        if (__builtin_expect(inside, 1)) {
#pragma unroll
            for (int g = 0; g < BATCH; ++g) raw[g] = load(index0 + (g0 + g) * step);
        } else {
            // next to an end of the tensor (which has at least four elements): loads that would leave it are moved inside, and
            // what they find there to where it belongs
            const int most = last_index + behind - 3;
#pragma unroll
            for (int g = 0; g < BATCH; ++g) {
                const int want = index0 + (g0 + g) * step;
                raw[g] = load(want < -before ? -before : want > most ? most : want);
            }
#pragma unroll
            for (int g = 0; g < BATCH; ++g) {
                const int want = index0 + (g0 + g) * step, front = -before - want, over = want - most;
#pragma unroll
                for (int r = 1; r < 4; ++r) {
                    const V v = raw[g];
                    raw[g][0] = over >= r ? v[1] : v[0];
                    raw[g][1] = front >= r ? v[0] : over >= r ? v[2] : v[1];
                    raw[g][2] = front >= r ? v[1] : over >= r ? v[3] : v[2];
                    raw[g][3] = front >= r ? v[2] : v[3];
                }
            }
        }
        if constexpr (!EXP) {                    // the scores themselves, -inf where there is no transition
#pragma unroll
            for (int g = 0; g < BATCH; ++g) {
                f32x4 w;
                const int ke = k_end(g0 + g);
#pragma unroll
                for (int k = 0; k < 4; ++k) w[k] = interior || valid(g0 + g, k, ke) ? Quad<TL>::get(raw[g], k) : DAGX_NEG_INF;
                *reinterpret_cast<f32x4 *>(dst + 4 * (g0 + g) * kPatchPitch) = w;
            }
            continue;
        }
        float lowest = 0.f;
        if (interior) {
#pragma unroll
            for (int g = 0; g < BATCH; ++g)
#pragma unroll
                for (int k = 0; k < 4; ++k) lowest = fminf(lowest, Quad<TL>::get(raw[g], k));
            if (__builtin_amdgcn_ballot_w64(lowest < -79.f) == 0) {
#pragma unroll
                for (int g = 0; g < BATCH; ++g) {
                    f32x4 w;
#pragma unroll
                    for (int k = 0; k < 4; ++k) w[k] = __builtin_ldexpf(fast_exp2(Quad<TL>::get(raw[g], k) * kLog2e), SHIFT);
                    *reinterpret_cast<f32x4 *>(dst + 4 * (g0 + g) * kPatchPitch) = w;
                }
                continue;
            }
        } else {
#pragma unroll
            for (int g = 0; g < BATCH; ++g) {
                const int ke = k_end(g0 + g);
#pragma unroll
                for (int k = 0; k < 4; ++k) lowest = fminf(lowest, valid(g0 + g, k, ke) ? Quad<TL>::get(raw[g], k) : 0.f);
            }
            if (__builtin_amdgcn_ballot_w64(lowest < -79.f) == 0) {
#pragma unroll
                for (int g = 0; g < BATCH; ++g) {
                    f32x4 w;
                    const int ke = k_end(g0 + g);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float v = __builtin_ldexpf(fast_exp2(Quad<TL>::get(raw[g], k) * kLog2e), SHIFT);
                        w[k] = valid(g0 + g, k, ke) ? v : 0.f;
                    }
                    *reinterpret_cast<f32x4 *>(dst + 4 * (g0 + g) * kPatchPitch) = w;
                }
                continue;
            }
        }
#pragma unroll
        for (int g = 0; g < BATCH; ++g) {
            f32x4 w;
            const int ke = k_end(g0 + g);
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = link_prob<SHIFT>(Quad<TL>::get(raw[g], k), valid(g0 + g, k, ke), tiny);
            *reinterpret_cast<f32x4 *>(dst + 4 * (g0 + g) * kPatchPitch) = w;
        }
    }
}
__device__ __forceinline__ void read_patch(Tile &t, const float *patch, int lane, int dir) {
    asm volatile("" ::: "memory");
    if (dir == 0) {
#pragma unroll
        for (int r = 0; r < kBlk; ++r) t.p[r] = patch[r * kPatchPitch + lane];
    } else {
#pragma unroll
        for (int r = 0; r < kBlk; r += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(patch + lane * kPatchPitch + kBlk - 4 - r);
            t.p[r] = v[3]; t.p[r + 1] = v[2]; t.p[r + 2] = v[1]; t.p[r + 3] = v[0];
        }
    }
    asm volatile("" ::: "memory");
}

// the patch as the float64 products want it: register 16 g + j, lane 16 k + o: row 4 j + k, position 16 g + o
__device__ __forceinline__ void read_patch_wide(Tile &t, const float *patch, int lane, int dir) {
    asm volatile("" ::: "memory");
    const int o = lane & 15, k = lane >> 4;
    const float *const src = dir == 0 ? patch + k * kPatchPitch + o : patch + o * kPatchPitch + kBlk - 1 - k;
    if (dir == 0) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int j = 0; j < 16; ++j) t.p[16 * g + j] = src[4 * j * kPatchPitch + 16 * g];
    } else {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int j = 0; j < 16; ++j) t.p[16 * g + j] = src[16 * g * kPatchPitch - 4 * j];
    }
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ double pow2_clamped_wide(int x, int floor_exp) {   // 2^x for x <= 0; 2^floor_exp (or 0: floor -1023) below
    const int c = x > floor_exp ? x : floor_exp;
    return __builtin_bit_cast(double, (unsigned long long)(unsigned)(c + 1023) << 52);
}
__device__ __forceinline__ float pow2_clamped(int x, int floor_exp) {   // 2^x for x <= 0; 2^floor_exp (or 0: floor -127) below
    const int c = x > floor_exp ? x : floor_exp;
    return __builtin_bit_cast(float, (unsigned)(c + 127) << 23);
}

}  // namespace dagx
