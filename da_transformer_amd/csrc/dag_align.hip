// Best alignment on gfx950: max-semiring sweep with back-pointers and an on-GPU backtrack.
//
//   A[t][j] = max_{i<j, j-i<=translen} fl32(A[t-1][i] + E[i][j]) + match[t][j]   (two fp32 roundings)
//   back[t][j] = the smallest i attaining the max; backtrack from (T_b-1, L_b-1).
//
// Two implementations:
//  * dag_align_chunks_kernel or dag_align_steps_kernel + dag_backtrack_kernel (L <= 1024): the sweep keeps E as 64x64 register
//    tiles, spread over the same pipeline of workgroups as the loss sweeps, and forms the sums by matrix instructions and one
//    three-way maximum per two (i, j) pairs -- four steps a stage, or, for few steps on many nodes, step by step
//    (align_in_chunks).  It stores the score table and the block of 64 nodes each cell's best predecessor lies in.  The
//    backtrack (a wave per sample walks, others may stage for it) then re-derives, for the T_b cells on the path only, the
//    lowest predecessor index attaining the stored maximum.
//  * dag_align_kernel: one workgroup per sample, thread <-> node j scanning its predecessors in
//    ascending order with a strict '>' (back-pointers in LDS when T*L fits, else in the caller's
//    workspace).  Handles any L <= 8192; the backtrack kernel uses the same code for the samples that the
//    pipeline gave up on.
// Both evaluate fl32(A + E) then + match, so their scores -- and therefore the paths -- are
// bit-identical to the torch-native rule.
#include "dag_chunks.h"

#include <atomic>

namespace dagx {

struct AlignArgs {
    const void *match; int64_t ms0, ms1, ms2;
    const void *links;
    const int64_t *out_len, *tgt_len;
    int B, T, L, translen;
    int64_t *path;
    int32_t *trace_ws;  // [B][T][L] when the LDS variant is not used
};

// One sample by one workgroup of NT threads; lds_a: 2*L floats, then (TRACE_LDS) T*L uint16.
template <typename TM, typename TL, int NT, bool TRACE_LDS>
__device__ __forceinline__ void align_one_sample(const AlignArgs &a, const int b, float *lds_a) {
    const int tid = threadIdx.x;
    const int L = a.L, T = a.T, translen = a.translen;
    const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
    const TM *match = static_cast<const TM *>(a.match) + (int64_t)b * a.ms0;
    const TL *links = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    int64_t *path = a.path + (int64_t)b * L;
    float *fprev = lds_a, *fcur = lds_a + L;
    uint16_t *tr_lds = reinterpret_cast<uint16_t *>(lds_a + 2 * (size_t)L);
    int32_t *tr_glb = TRACE_LDS ? nullptr : a.trace_ws + (int64_t)b * T * L;

    for (int j = tid; j < L; j += NT) path[j] = -1;
    const bool ok = Tb >= 1 && Lb >= 1 && Tb <= T && Lb <= L && Tb <= Lb;
    if (!ok) return;
    const int slack = Lb - Tb;

    const float first = to_float(match[0]);
    for (int j = tid; j < L; j += NT) fprev[j] = (j == 0) ? first : DAGX_NEG_INF;
    __syncthreads();

    // A team of kTeam lanes <-> node j of the band; the team's lanes deal the predecessors i among themselves
    // (lane q takes i = ilo + q, ilo + q + kTeam, ...), R of them in flight per lane, and merge their
    // (best score, lowest index that has it) pairs by shuffles.  Nodes go to the teams round robin, which mixes
    // nodes with few and with many predecessors in every team.  Cells outside the band are never on a path:
    // their trace entries stay unwritten.
    constexpr int kTeam = 8, R = 8;
    const int team = tid / kTeam, sub = tid % kTeam;
    const unsigned rs = (unsigned)(translen - 1);   // E[i][j-i-1] sits at links[i*(translen-1) + j-1]: 32-bit offsets
    for (int t = 1; t < Tb; ++t) {
        const int jhi = slack + t;
        for (int j = tid; j < L; j += NT)
            if (j < t || j > jhi) fcur[j] = DAGX_NEG_INF;
        for (int j = t + team; j <= jhi; j += NT / kTeam) {
            const float mj = to_float(match[(int64_t)t * a.ms1 + (int64_t)j * a.ms2]);
            int ilo = j - translen; if (ilo < t - 1) ilo = t - 1;
            float best = DAGX_NEG_INF;
            int arg = ilo;
            const unsigned o_last = (unsigned)(j - 1) * (unsigned)translen;   // the offset of i = j-1, the largest
            unsigned o = (unsigned)(ilo + sub) * rs + (unsigned)(j - 1);
            for (int i0 = ilo + sub; i0 < j; i0 += kTeam * R, o += kTeam * R * rs) {
                float e[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const unsigned oc = o + (unsigned)(r * kTeam) * rs;
                    e[r] = to_float(links[oc < o_last ? oc : o_last]);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int i = i0 + r * kTeam;
                    const float x = i < j ? fprev[i < j ? i : j - 1] + e[r] : DAGX_NEG_INF;   // (index clamped: read, then selected)
                    if (x > best) { best = x; arg = i; }
                }
            }
#pragma unroll
            for (int w = kTeam / 2; w > 0; w >>= 1) {
                const float bo = __shfl_xor(best, w, kWave);
                const int ao = __shfl_xor(arg, w, kWave);
                if (bo > best || (bo == best && ao < arg)) { best = bo; arg = ao; }
            }
            if (sub == 0) {
                fcur[j] = best + mj;
                if (TRACE_LDS) tr_lds[(size_t)t * L + j] = (uint16_t)arg;
                else tr_glb[(int64_t)t * L + j] = arg;
            }
        }
        __syncthreads();
        float *sw = fprev; fprev = fcur; fcur = sw;
    }

    if (tid == 0 && fprev[Lb - 1] > DAGX_NEG_INF) {
        int j = Lb - 1;
        for (int t = Tb - 1; t >= 0; --t) {
            path[j] = t;
            if (t > 0) j = TRACE_LDS ? (int)tr_lds[(size_t)t * L + j] : tr_glb[(int64_t)t * L + j];
        }
    }
}

template <typename TM, typename TL, int NT, bool TRACE_LDS>
__global__ __launch_bounds__(NT) void dag_align_kernel(AlignArgs a) {
    extern __shared__ __align__(16) float lds_a[];
    align_one_sample<TM, TL, NT, TRACE_LDS>(a, blockIdx.x, lds_a);
}


// ================================================================================================
// Tile-resident max-plus sweep
// ================================================================================================

// The sums of max-plus on the matrix cores: v_mfma_f32_4x4x1_16b with a second operand of ones and the tile's registers as the
// third is cells[row] + P[row][lane] for four rows, one rounding each (1 * x is exact: the bits of v_add_f32, subnormals
// and infinities among them).  256 sums take 8.2 cycles of a SIMD and four v_add_f32_dpp 18; the maxima, a three-way one for two
// sums at 4.5 cycles, are all that vector instructions have left to do.  A change between matrix and vector instructions costs
// a SIMD about 6.5 cycles, hence four of the former and eight of the latter at a time, sixteen registers of sums.  Four steps of a
// tile, ns, on a wave alone and for each of two that share a SIMD, all in one run: four at a time 585 and 546, one at a time 824 and 690, eight
// at a time, with sixteen registers more, 560 and 517; in two DPP sums and a maximum for every two rows 980 and 782.
//
// d = cells[4 ABID + i] + t.p[ROW + i] for i < 4; CBSZ 4: the cells of all 64 lanes are candidates, 3: those of a lane's own half
template <int CBSZ, int ABID, int ROW>
__device__ __forceinline__ f32x4 four_sums(const Tile &t, float cells) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(cells, 1.f, f32x4{t.p[ROW], t.p[ROW + 1], t.p[ROW + 2], t.p[ROW + 3]}, CBSZ, ABID, 0);
}
// (a maximum does not round: neither three-way ones nor the order change anything)
__device__ __forceinline__ void raise(float &b0, float &b1, f32x4 d) {
    b0 = fmaxf(fmaxf(d[0], d[1]), b0);
    b1 = fmaxf(fmaxf(d[2], d[3]), b1);
}
// (batches stay as they are written)
__device__ __forceinline__ void batch_end() { __builtin_amdgcn_sched_barrier(0); }

// max_{r<64} (cells[r] + tile.p[r]) for two steps; lane r holds cells[r]
__device__ __forceinline__ void tile_maxplus2(const Tile &t, float x, float y, float &out0, float &out1) {
    float b0 = DAGX_NEG_INF, b1 = DAGX_NEG_INF, c0 = DAGX_NEG_INF, c1 = DAGX_NEG_INF;
    auto rows8 = [&](auto at) __attribute__((always_inline)) {
        constexpr int K = decltype(at)::value;
        const f32x4 d0 = four_sums<4, K, 4 * K>(t, x), d1 = four_sums<4, K, 4 * K>(t, y);
        const f32x4 d2 = four_sums<4, K + 1, 4 * K + 4>(t, x), d3 = four_sums<4, K + 1, 4 * K + 4>(t, y);
        batch_end();
        raise(b0, b1, d0); raise(c0, c1, d1); raise(b0, b1, d2); raise(c0, c1, d3);
        batch_end();
    };
    rows8(std::integral_constant<int, 0>{}); rows8(std::integral_constant<int, 2>{});
    rows8(std::integral_constant<int, 4>{}); rows8(std::integral_constant<int, 6>{});
    rows8(std::integral_constant<int, 8>{}); rows8(std::integral_constant<int, 10>{});
    rows8(std::integral_constant<int, 12>{}); rows8(std::integral_constant<int, 14>{});
    out0 = fmaxf(b0, b1); out1 = fmaxf(c0, c1);
}

// {x, y} -> x: rows {x0 y0 x2 y2} of sixteen lanes, y: rows {x1 y1 x3 y3}
__device__ __forceinline__ void swap_rows(float &x, float &y) {
    const u32x2 s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y), false, false);
    const unsigned a = s[0], b = s[1];
    x = __builtin_bit_cast(float, a); y = __builtin_bit_cast(float, b);
}
// b0, b1 raised by sixteen rows of one step
template <int CBSZ, int ABID, int ROW>
__device__ __forceinline__ void rows16(const Tile &t, float cells, float &b0, float &b1) {
    const f32x4 d0 = four_sums<CBSZ, ABID, ROW>(t, cells), d1 = four_sums<CBSZ, ABID + 1, ROW + 4>(t, cells);
    const f32x4 d2 = four_sums<CBSZ, ABID + 2, ROW + 8>(t, cells), d3 = four_sums<CBSZ, ABID + 3, ROW + 12>(t, cells);
    batch_end();
    raise(b0, b1, d0); raise(b0, b1, d1); raise(b0, b1, d2); raise(b0, b1, d3);
    batch_end();
}
// max_i (a[i] + P[i][lane]) over a triangle as fold_triangle leaves it; `upper`: lanes 32..63
__device__ __forceinline__ float triangle_maxplus(const Tile &t, float a, bool upper) {
    float even = a, crossed = a;
    swap_rows(even, crossed);                  // rows {0,0,2,2} and {1,1,3,3} of a
    float b0 = DAGX_NEG_INF, b1 = DAGX_NEG_INF, c0 = DAGX_NEG_INF, c1 = DAGX_NEG_INF;
    swap_halves(crossed, even);                // rows {1,1,0,0}
    rows16<3, 0, 32>(t, crossed, c0, c1);
    float other = fmaxf(c0, c1), square = other;
    rows16<3, 0, 0>(t, a, b0, b1);
    swap_halves(square, other);                // (the square's two halves, for the upper lanes)
    rows16<3, 4, 16>(t, a, b0, b1);
    square = fmaxf(square, other);
    return fmaxf(fmaxf(b0, b1), upper ? square : DAGX_NEG_INF);
}

// bytes per row of the source-block table (rows padded to 16 bytes)
__host__ __device__ static inline int srcblk_pitch(int L) { return (L + 15) & ~15; }

// Contiguous grouping of the position blocks [0, NBb) into at most C groups of at most kTileCap tiles,
// minimising the largest group.  gstart[g] .. gstart[g+1] are the blocks of group g (empty groups last).
__device__ __host__ inline int partition_blocks(int NBb, int W, int C, int *gstart) {
    int best_cap = kTileCap;
    for (int cap = 1; cap <= kTileCap; ++cap) {
        int groups = 1, sum = 0; bool ok = true;
        for (int Jb = 0; Jb < NBb; ++Jb) {
            int c = Jb - tile_ilo(Jb, W) + 1;
            if (c > cap) { ok = false; break; }
            if (sum + c > cap) { ++groups; sum = 0; }
            sum += c;
        }
        if (ok && groups <= C) { best_cap = cap; break; }
    }
    int g = 0, sum = 0;
    gstart[0] = 0;
    for (int Jb = 0; Jb < NBb; ++Jb) {
        int c = Jb - tile_ilo(Jb, W) + 1;
        if (sum + c > best_cap && sum > 0) { ++g; if (g < C) gstart[g] = Jb; sum = 0; }
        sum += c;
    }
    int used = g + 1;
    for (int q = used; q <= C; ++q) gstart[q] = NBb;
    return used;
}

struct AlignTileArgs {
    const void *match; int64_t ms0, ms1, ms2;
    const void *links;
    const int64_t *out_len, *tgt_len;
    int B, T, L, translen;
    float *table;     // [B][T][L] best score of every cell, by node
    unsigned char *srcblk;   // [B][T][pitch] block of 64 nodes that holds the best predecessor of every cell (the lowest such block); 16-byte aligned rows
    int *sync;        // [0] ticket counter, [16 + b*C + group] progress
    int *flags;       // [B] set when the pipeline gave up on a sample
    int C;
    int mcap;         // match row read at step s: min(s, mcap) (T-1 for the alignment: every step its own row)
    int decode;       // Viterbi decoding: every sample runs all T steps (tgt_len is not read) and no cell is
                      // pruned for being too far from the last node -- a path may end at any step
    ChunkPlan<1> plan;   // gtab[NBb][g] = first block of group g, and how its tiles are dealt to its waves
};

// The pipeline of the loss sweeps (sweep_chunks_group: stages of four steps, tickets, one-way hand-over through the table
// with agent-scope accesses, bounded waits), in the (max, +) semiring and without any rescaling: the table holds the plain
// fp32 scores, and a foreign block's rows are copied straight to where the tiles read them.  A maximum does not round and
// sums are formed as they are step by step, so that scores and source blocks do not depend on the order: of several
// blocks with the best predecessor the lowest one counts (runs in the order of the blocks, then the block itself; a later
// one replaces an earlier one only if it is larger).
//
// What bounds the stages is the tiles' sums and maxima, 1 300 cycles of a SIMD for four steps of a tile (a SIMD gives its cycles
// to matrix or to vector instructions, so that two waves that share one gain hardly anything), and the walks.
//
// SPACING (dag_chunks.h): a tile is nearly as much work as the walk here, so that where the walk bounds the stages and SIMDs
// have time to spare -- small graphs, or hardly more than one block to a group -- two stages a block are shorter
// (alignment with SPACING 1 and 2: B = 64, L = 256, T = 64 77.0 and 70.5 us; B = 64, L = 320, T = 48 69.9 and 66.9; B = 40, L = 400, T = 60 91.2
// and 90.8); where the tiles bound them every stage more costs (B = 64, L = 512, T = 64 109.4 and 112.6).
template <typename TM, typename TL, int SPACING>
__global__ __launch_bounds__(kTileWaves * kWave) void dag_align_chunks_kernel(AlignTileArgs a) {
    extern __shared__ __align__(16) float lds_raw[];
    __shared__ int gstart[16];
    __shared__ int s_ticket, s_abort;

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int C = a.C;
    if (tid == 0) { s_ticket = atomicAdd(a.sync, 1); s_abort = 0; }
    __syncthreads();
    const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    const int B8 = (a.B + 7) & ~7;
    // first group 0 of every sample, then every group 1, ... (see the loss sweep kernel: producers hold smaller tickets,
    // and what the dispatcher reaches last are consumers); the groups of a sample are a multiple of 8 tickets apart
    const int g = ticket / B8;
    const int b = ((ticket / 8) % (B8 / 8)) * 8 + (ticket % 8);
    if (g >= C || b >= a.B) return;

    const int L = opaque_uniform(a.L), T = a.T, translen = a.translen;
    const int Lb = (int)a.out_len[b], Tb = a.decode ? T : (int)a.tgt_len[b];
    if (!(Tb >= 1 && Lb >= 1 && Tb <= T && Lb <= L && (a.decode || Tb <= Lb))) return;   // the backtrack sees the lengths too
    const TM *match = static_cast<const TM *>(a.match) + (int64_t)b * a.ms0;
    const TL *links = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    float *table = a.table + (int64_t)b * T * L;
    const int spitch = srcblk_pitch(L);
    unsigned char *srcblk = a.srcblk + (int64_t)b * T * spitch;
    int *prog = a.sync + 16 + b * C;

    const int slack = a.decode ? L : Lb - Tb;
    const int NBb = (Lb + kBlk - 1) / kBlk;
    const int W = (translen + kBlk - 1) / kBlk;
    if (tid <= C) gstart[tid] = a.plan.gtab[0][NBb][tid];
    __syncthreads();
    const int jb0 = __builtin_amdgcn_readfirstlane(gstart[g]), jb1 = __builtin_amdgcn_readfirstlane(gstart[g + 1]);
    int last_group = 0;
    for (int q = 0; q < C; ++q) if (gstart[q + 1] > gstart[q]) last_group = q;
    last_group = __builtin_amdgcn_readfirstlane(last_group);
    if (jb0 >= jb1) return;
    const int nblk = jb1 - jb0;
    const int flo = tile_ilo(jb0, W);
    const bool producer = g < last_group, consumer = flo < jb0;
    const AlignLds o = align_lds(jb0, nblk, W, SPACING);
    if (nblk > kChunkBlocks || o.total * 4 > kChunkLdsBytes) {   // cannot happen with the host's partition
        if (tid == 0) { a.flags[b] = 1; store_agent(prog + g, 1 << 30); }
        return;
    }
    const bool owner = wave < nblk;               // this wave walks block jb0 + wave
    const int helpers = kTileWaves - nblk;
    const TileDeal deal = a.plan.deal[0][NBb][g];
    const WaveTiles t = plan_wave<SPACING>(deal, jb0, nblk, W, 0, wave, lane);
    // (Progress words as in the loss sweeps.)
    if (consumer) {
        if (wave == 0)
            for (int spins = 0; spins < kSpinLimit && __builtin_amdgcn_readfirstlane(load_agent(prog)) < 1; ++spins) __builtin_amdgcn_s_sleep(8);
        __syncthreads();
    }
    const unsigned lds_base = (unsigned)reinterpret_cast<uintptr_t>(lds_raw);
    float *const patch = lds_raw + wave * (kBlk * kPatchPitch);
    const int last_index = L * translen - 1;
    auto elements = [&](const int samples) { const int64_t n = (int64_t)samples * L * translen; return n < (1 << 28) ? (int)n : 1 << 28; };
    const int before = elements(b), behind = elements(a.B - 1 - b);
    auto stage = [&](Tile &tile, const int u) __attribute__((always_inline)) {
        stage_tile<TL, 0, false>(patch, links, t.I[u], jb0 + t.q[u], lane, 0, Lb, translen, last_index, before, behind, 0.f);
        read_patch(tile, patch, lane, 0);
    };
    Tile t0, t1, t2;
    if (t.ok[0] || t.adjacent) stage(t0, 0);
    if (t.ok[1]) stage(t1, 1);
    if (t.ok[2] || owner) stage(t2, 2);
    if (owner) fold_triangle(t2, lane);
    __syncthreads();   // every wave is done with its transpose patch: the LDS now holds the buffers of the stages
    if (producer && g == 0 && tid == 0) store_agent(prog, 1);

    int *const lds_i = reinterpret_cast<int *>(lds_raw);
    int *const published_by = lds_i + o.both;
    if (tid == 0) *published_by = 0;
    const int D = o.depth;
    const char *match_c = reinterpret_cast<const char *>(match);
    const int ms1 = opaque_uniform((int)a.ms1), ms2 = opaque_uniform((int)a.ms2);   // the host checked that match indices fit 32 bits
    // step 0: node 0 holds match[0][0] (even if that is -inf), everything else -inf
    const float m0 = to_float(match[0]);
    if (owner) {
        const int p = (jb0 + wave) * kBlk + lane;
        const float v = p == 0 ? m0 : DAGX_NEG_INF;
        lds_raw[o.eb + (jb0 - flo + wave) * D * 256 + lane] = v;
        if (p < Lb) store_agent(table + p, v);
    }
    const unsigned long long table_u = uniform_address(table);
    char *const table_c = reinterpret_cast<char *>(table), *const srcblk_c = reinterpret_cast<char *>(srcblk);
    const int NC = (Tb - 1 + kChunk - 1) / kChunk;  // chunks of steps 1 .. T_b-1
    const int last_row = opaque_uniform(a.mcap < Tb - 1 ? a.mcap : Tb - 1);
    auto opaque_lane = [&] { int x = tid & (kWave - 1); asm volatile("" : "+v"(x)); return x; };
    // a block's chunks with a cell in the band (4c+1 .. 4c+4), and its chunks as a source (4c .. 4c+3)
    auto dest_lo = [&](const int J) { return 16 * J - 1 - (slack >> 2); };
    auto dest_hi = [&](const int J) { return 16 * J + 15; };
    auto src_lo = [&](const int I) { return 16 * I - ((slack + 3) >> 2); };

    // ---- the foreign blocks whose table rows this wave fetches ----
    int f_blk[kForeign], f_first, f_count;
    wave_foreign(deal, wave, f_first, f_count);
#pragma unroll
    for (int u = 0; u < kForeign; ++u) f_blk[u] = u < f_count ? flo + f_first + u : -1;
    // table rows of steps 4c .. 4c+3 of a foreign block (complete: 64 nodes) to slot sl of its cells: sixteen bytes a lane
    auto request_rows = [&](const int I, const int c, const int sl, const int lane) __attribute__((always_inline)) {
        const int s = kChunk * c + (lane >> 4), row = s < Tb ? s : Tb - 1;
        dma_dwordx4_agent_u(lds_base + (unsigned)(o.eb + ((I - flo) * D + sl) * 256) * 4u, table_u, (unsigned)(row * L + I * kBlk + 4 * (lane & 15)) * 4u);
    };

    // ---- the stages ----
    const int first_stage = consumer ? -2 : -1, end_stage = NC - 1 + SPACING * (nblk - 1);
    const int *below = prog + (g > 0 ? g - 1 : 0);
    // stages in which a tile's block takes part, and those in which the tile's source has a cell in the band
    int t_from[kTilesPerWave], t_to[kTilesPerWave], t_src_from[kTilesPerWave], t_src_to[kTilesPerWave], t_shift[kTilesPerWave], t_cells[kTilesPerWave];
#pragma unroll
    for (int u = 0; u < kTilesPerWave; ++u) {
        const int J = jb0 + t.q[u], at = SPACING * t.q[u] - 1;               // chunk = stage - at
        t_from[u] = at + (dest_lo(J) > 0 ? dest_lo(J) : 0);
        t_to[u] = t.ok[u] ? at + (dest_hi(J) < NC - 1 ? dest_hi(J) : NC - 1) : -100;
        t_src_from[u] = at + src_lo(t.I[u]); t_src_to[u] = at + dest_hi(t.I[u]);
        t_shift[u] = (((-at) % D) + D) % D;
        t_cells[u] = o.eb + (t.I[u] - flo) * D * 256;
    }
    if (NC == 0) return;
    __syncthreads();

    auto stages = [&](auto walks, auto fetches) __attribute__((always_inline)) {
        constexpr bool WALKS = decltype(walks)::value, FETCHES = decltype(fetches)::value;
        int slot_own = 0, seen = 0, requested = first_stage - 1, ring = ((first_stage % D) + D) % D;
        auto next_slot = [&](const int x) { return x + 1 == D ? 0 : x + 1; };
        const int J = jb0 + wave, first = J * kBlk, own_src = jb0 - flo + wave, ilo = tile_ilo(J, W);
        float e = WALKS && J == 0 && lane == 0 ? m0 : DAGX_NEG_INF;          // the last step's scores
        float mt[kChunk] = {0.f, 0.f, 0.f, 0.f};                             // the next chunk's match rows
        TM raw[kChunk];
        auto load_match = [&](const int c, const int lane) __attribute__((always_inline)) {
            const int p = first + lane, pc = p < Lb ? p : Lb - 1, s0 = kChunk * c + 1;
            const unsigned lane_off = (unsigned)(pc * ms2) * (unsigned)sizeof(TM);
#pragma unroll
            for (int k = 0; k < kChunk; ++k)
                raw[k] = *reinterpret_cast<const TM *>(match_c + (unsigned)((s0 + k < last_row ? s0 + k : last_row) * ms1) * (unsigned)sizeof(TM) + lane_off);
        };
        auto convert_match = [&] {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) mt[k] = to_float(raw[k]);
        };
        // a tile's best of four steps into the best so far (this lane's place in the cells of four steps, 64 each)
        auto take = [&](const Tile &tile, const float *cells, const int I, float (&best)[kChunk], int (&from)[kChunk]) __attribute__((always_inline)) {
            float cell[kChunk];
#pragma unroll
            for (int k = 0; k < kChunk; ++k) cell[k] = cells[k * kBlk];
#pragma unroll
            for (int k = 0; k < kChunk; k += 2) {
                float x[2];
                tile_maxplus2(tile, cell[k], cell[k + 1], x[0], x[1]);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool up = x[h] > best[k + h];
                    best[k + h] = up ? x[h] : best[k + h]; from[k + h] = up ? I : from[k + h];
                }
            }
        };
        for (int tau = first_stage; tau <= end_stage; ++tau) {
            const int par = tau & 1;
            const int lane = opaque_lane();
            // (chunk tau + 2 of the foreign blocks, with SPACING 1 tau + 1 of the block below)
            const bool bring = FETCHES && f_blk[0] >= 0 && tau + SPACING < NC;
            int published = 0;
            if (bring) published = load_agent(below);
            // (as in the loss sweeps; with SPACING 2 the last block's wave alone: the other blocks are two stages ahead of it)
            auto publish = [&]() __attribute__((always_inline)) {
                const int n = tau - SPACING * (nblk - 1);      // chunks of the last block
                if (!producer || wave < nblk - (SPACING == 1 ? 2 : 1) || n < 0 || n >= NC) return;
                wait_vmem_all();
                int both = 1;
                if (SPACING == 1 && nblk > 1) {
                    if (lane == 0) both = __hip_atomic_fetch_add(published_by, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & 1;
                }
                if (lane == 0 && both) store_agent(prog + g, 2 + n);
            };
            // ---------------- walk my block through chunk tau - SPACING wave ----------------
            if (WALKS) {
                const int c = tau - SPACING * wave;
                const bool more = c >= -1 && c + 1 < NC, live = c >= 0 && c < NC && c >= dest_lo(J) && c <= dest_hi(J);
                float best[kChunk] = {DAGX_NEG_INF, DAGX_NEG_INF, DAGX_NEG_INF, DAGX_NEG_INF};
                int from[kChunk] = {ilo, ilo, ilo, ilo};
                if (live) {
                    __builtin_amdgcn_s_setprio(3);
                    if (J > (SPACING == 1 ? ilo + 1 : 0)) {
#pragma unroll 1
                        for (int u = 0; u < t.run_count; ++u) {
                            const int at = (t.run_first + u) * 2 + (par ^ 1);
                            const f32x4 x = *reinterpret_cast<const f32x4 *>(lds_raw + o.part + at * 256 + lane * 4);
                            const int y = lds_i[o.from + at * 64 + lane];
#pragma unroll
                            for (int k = 0; k < kChunk; ++k) {
                                const float xk = x[k];
                                const bool up = xk > best[k];
                                best[k] = up ? xk : best[k]; from[k] = up ? (y >> (8 * k)) & 255 : from[k];
                            }
                        }
                    }
                    if (SPACING == 1 && J > 0 && c >= src_lo(J - 1) && c <= dest_hi(J - 1))   // what block J - 1 sends
                        take(t0, lds_raw + o.eb + ((own_src - 1) * D + slot_own) * 256 + lane, J - 1, best, from);
                }
                if (more) load_match(c + 1, lane);
                if (c >= 0 && c < NC) {
                    float *const cells = lds_raw + o.eb + own_src * D * 256 + lane;
                    float *const cells_next = cells + next_slot(slot_own) * 256;
                    float *const cells_this = cells + slot_own * 256;
                    const int s0 = kChunk * c + 1;
                    float v[kChunk];
                    if (live) {
                        const int d0 = first + lane - s0;
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            const float x = triangle_maxplus(t2, e, lane >= 32);
                            const bool up = x > best[k];
                            best[k] = up ? x : best[k]; from[k] = up ? J : from[k];
                            // in the band: s <= p <= slack + s; the second (and last) rounding of the cell
                            e = (unsigned)(d0 - k) <= (unsigned)slack ? best[k] + mt[k] : DAGX_NEG_INF;
                            v[k] = e;
                            if (k < kChunk - 1) cells_this[kBlk * (k + 1)] = e; else cells_next[0] = e;
                            if (k == 0) publish();
                        }
                        __builtin_amdgcn_s_setprio(0);
                    } else {
                        publish();
                        e = DAGX_NEG_INF;
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            v[k] = e;
                            if (k < kChunk - 1) cells_this[kBlk * (k + 1)] = e; else cells_next[0] = e;
                        }
                    }
                    if (more) convert_match();   // (in front of the stores: what it waits for is older than they)
                    else wait_vmem_all();
                    // into the tables
                    const int steps = Tb - s0 < kChunk ? Tb - s0 : kChunk;
                    if (first + lane < Lb) {
                        char *row = table_c + (unsigned)(s0 * L) * 4u, *srow = srcblk_c + (unsigned)(s0 * spitch);
                        const unsigned at = (unsigned)(first + lane);
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            if (k >= steps) break;
                            store_agent(reinterpret_cast<float *>(row + at * 4u), v[k]);
                            *reinterpret_cast<unsigned char *>(srow + at) = (unsigned char)from[k];
                            row += L * 4; srow += spitch;
                        }
                    }
                    slot_own = next_slot(slot_own);
                }
                else {
                    publish();
                    if (more) convert_match();
                    else if (SPACING == 1 && c == NC) wait_vmem_all();
                }
            }
            // ---------------- what my tiles' blocks (q of the group) receive in chunk tau + 1 - SPACING q ------
            if (t.count > 0) {
                float best[kChunk] = {DAGX_NEG_INF, DAGX_NEG_INF, DAGX_NEG_INF, DAGX_NEG_INF};
                int from[kChunk] = {0, 0, 0, 0};
                auto product = [&](const int u, const Tile &tile) __attribute__((always_inline)) {
                    if (!(tau >= t_from[u] && tau <= t_to[u])) return;
                    if (t.start[u]) {
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) { best[k] = DAGX_NEG_INF; from[k] = 0; }
                    }
                    if (tau >= t_src_from[u] && tau <= t_src_to[u]) {
                        int sl = ring + t_shift[u]; sl -= sl >= D ? D : 0;
                        take(tile, lds_raw + t_cells[u] + sl * 256 + lane, t.I[u], best, from);
                    }
                    if (t.end[u]) {
                        const int at = t.run[u] * 2 + par;
                        *reinterpret_cast<f32x4 *>(lds_raw + o.part + at * 256 + lane * 4) = f32x4{best[0], best[1], best[2], best[3]};
                        lds_i[o.from + at * 64 + lane] = from[0] | from[1] << 8 | from[2] << 16 | from[3] << 24;
                    }
                };
                if (SPACING == 2 || !WALKS) product(0, t0);
                product(1, t1);
                if (!WALKS) product(2, t2);
            }
            // ---------------- table rows of foreign blocks: requested a stage ago if they were published by then ----------------
            if (bring) {
                published = __builtin_amdgcn_readfirstlane(published);
                if (published > seen) seen = published;
                auto request = [&](const int stage) __attribute__((always_inline)) {   // what a stage brings in
#pragma unroll
                    for (int u = 0; u < kForeign; ++u) {
                        if (f_blk[u] < 0) break;
                        const int c = stage + (SPACING == 1 && f_blk[u] == jb0 - 1 ? 1 : 2);
                        int sl = ring + c - tau; sl -= sl >= D ? D : 0;
                        if (SPACING == 2 || (c >= 0 && c < NC)) request_rows(f_blk[u], c, sl, lane);
                    }
                    requested = stage;
                };
                if (requested < tau) {
                    int spins = 0;
                    while (seen < tau + SPACING + 3) {
                        __builtin_amdgcn_s_sleep(1);
                        seen = __builtin_amdgcn_readfirstlane(load_agent(below));
                        if (++spins > kSpinLimit) { s_abort = 1; break; }
                    }
                    if (seen >= tau + SPACING + 3) request(tau);
                }
                wait_vmem_all();
                if (tau + 1 + SPACING < NC && seen >= tau + SPACING + 4) request(tau + 1);
            }
            ring = next_slot(ring);
            __syncthreads();
            if (consumer && __builtin_amdgcn_readfirstlane(s_abort)) return;
        }
    };
    if (owner && helpers == 0) stages(std::true_type{}, std::true_type{});
    else if (owner) stages(std::true_type{}, std::false_type{});
    else stages(std::false_type{}, std::true_type{});
    if (producer) {
        wait_vmem_all();
        __syncthreads();
        if (tid == 0) store_agent(prog + g, 2 + NC);
    }
    if (consumer && __builtin_amdgcn_readfirstlane(s_abort)) {   // a producer never showed up: the sample is done again, and consumers go on
        wait_vmem_all();
        if (tid == 0) { a.flags[b] = 1; store_agent(prog + g, 1 << 30); }
    }
}

__device__ __forceinline__ float max3(float a, float b, float c) {
    float d;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

// max_{r<64} (a[r] + tile.p[r]); lane r holds a[r]
__device__ __forceinline__ float tile_maxplus(const Tile &t, float a) {
    float b0 = DAGX_NEG_INF, b1 = DAGX_NEG_INF;
    rows16<4, 0, 0>(t, a, b0, b1);
    rows16<4, 4, 16>(t, a, b0, b1);
    rows16<4, 8, 32>(t, a, b0, b1);
    rows16<4, 12, 48>(t, a, b0, b1);
    return fmaxf(b0, b1);
}

// The same sweep step by step, for few steps on many nodes (launch_align_sweep): the groups follow each other a few steps
// apart instead of a few stages, and a step waits for nobody but the group below.
//
// One tile of scores: t.p[r] = E(node 64 I + r -> node 64 J + lane), -inf where there is no transition; sixteen loads in
// flight (clamped to element 0).
template <typename TL>
__device__ __forceinline__ void load_scores(Tile &t, const TL *links, int I, int J, int lane, int Lb, int translen) {
    const int dd = (J - I) * kBlk - 1;   // distance: dd + lane - r
    const char *const lbase = reinterpret_cast<const char *>(links);
    // every (row, lane) of the tile is a transition of the sample (wave-uniform)
    const bool interior = J > I && dd + kBlk - 1 < translen && J * kBlk + kBlk - 1 < Lb;
    constexpr int CH = 16;
    const int p_out = J * kBlk + lane;
    const int base = I * kBlk * translen + dd + lane;
    const int step = translen - 1;
    const bool col_ok = p_out < Lb;
    TL raw[2][CH];
    auto request = [&](const int c, TL (&dst)[CH]) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < CH; ++r) {
            const int d = dd + lane - (c + r);
            const bool valid = col_ok && d >= 0 && d < translen;
            dst[r] = *reinterpret_cast<const TL *>(lbase + (interior || valid ? (unsigned)(base + (c + r) * step) * (unsigned)sizeof(TL) : 0u));
        }
    };
    request(0, raw[0]);
#pragma unroll
    for (int k = 0; k < kBlk / CH; ++k) {
        const int c = k * CH;
        if (k + 1 < kBlk / CH) request(c + CH, raw[(k + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        const TL (&e)[CH] = raw[k & 1];
        if (interior) {
#pragma unroll
            for (int r = 0; r < CH; ++r) t.p[c + r] = to_float(e[r]);
        } else {
            bool valid[CH];
#pragma unroll
            for (int r = 0; r < CH; ++r) {
                const int d = dd + lane - (c + r);
                valid[r] = col_ok && d >= 0 && d < translen;
            }
#pragma unroll
            for (int r = 0; r < CH; ++r) t.p[c + r] = valid[r] ? to_float(e[r]) : DAGX_NEG_INF;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <typename TM, typename TL>
__global__ __launch_bounds__(kTileWaves * kWave) void dag_align_steps_kernel(AlignTileArgs a) {
    __shared__ float abuf[2][kMaxBlocksFast][kBlk];   // scores of the previous / next step, by node
    // tile results: the tiles of an owned block lie in consecutive rows that start at a multiple of eight, and the rows
    // behind them, up to the next multiple of eight, hold -inf for good: the owner reads whole eights without a test
    constexpr int kPartRows = kTileCap + 7 * kMaxBlocksFast;
    __shared__ float part[kPartRows][kBlk];
    // landing areas of the asynchronous global -> LDS copies (one slot per consuming wave), double-buffered by step parity
    __shared__ unsigned stage_m[2][kTileWaves][2][kBlk];   // match rows of the wave's own blocks (raw elements)
    __shared__ float stage_f[2][kTileWaves][2][kBlk];      // table rows of the wave's foreign blocks
    __shared__ int stage_p[2][kBlk];                        // snapshots of the progress word of the group below
    __shared__ int gstart[kTileCap + 2];
    __shared__ int s_ticket, s_abort;

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int C = a.C;
    if (tid == 0) { s_ticket = atomicAdd(a.sync, 1); s_abort = 0; }
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(s_ticket);
    const int B8 = (a.B + 7) & ~7;
    // first group 0 of every sample, then every group 1, ... (see the loss sweep kernel: producers hold smaller tickets,
    // and what the dispatcher reaches last are consumers); the groups of a sample are a multiple of 8 tickets apart
    const int g = k / B8;
    const int b = ((k / 8) % (B8 / 8)) * 8 + (k % 8);
    if (g >= C || b >= a.B) return;

    const int L = a.L, T = a.T, translen = a.translen;
    const int Lb = (int)a.out_len[b], Tb = a.decode ? T : (int)a.tgt_len[b];
    if (!(Tb >= 1 && Lb >= 1 && Tb <= T && Lb <= L && (a.decode || Tb <= Lb))) return;   // the backtrack sees the lengths too
    const TM *match = static_cast<const TM *>(a.match) + (int64_t)b * a.ms0;
    const TL *links = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    float *table = a.table + (int64_t)b * T * L;
    const int spitch = srcblk_pitch(L);
    unsigned char *srcblk = a.srcblk + (int64_t)b * T * spitch;
    int *prog = a.sync + 16 + b * C;

    const int slack = a.decode ? L : Lb - Tb;
    const int mcap = a.mcap;
    const int NBb = (Lb + kBlk - 1) / kBlk;
    const int W = (translen + kBlk - 1) / kBlk;
    if (tid <= C) gstart[tid] = a.plan.gtab[0][NBb][tid];
    __syncthreads();
    const int jb0 = __builtin_amdgcn_readfirstlane(gstart[g]), jb1 = __builtin_amdgcn_readfirstlane(gstart[g + 1]);
    int last_group = 0;
    for (int q = 0; q < C; ++q) if (gstart[q + 1] > gstart[q]) last_group = q;
    last_group = __builtin_amdgcn_readfirstlane(last_group);
    if (jb0 >= jb1) return;
    const int nblk = jb1 - jb0;
    const int flo = tile_ilo(jb0, W);
    const bool producer = g < last_group;
    const bool consumer = flo < jb0;

    int ntile = 0;
    for (int Jb = jb0; Jb < jb1; ++Jb) ntile += Jb - tile_ilo(Jb, W) + 1;
    // The last wave is the fetcher (it works one step ahead of the others, see fetch_step) and takes tiles only when the others cannot
    // hold them all; the tiles are dealt out evenly, the odd ones first to wave 3 (the fetcher's SIMD).
    const int nwork = ntile <= kTilesPerWave * (kTileWaves - 1) ? kTileWaves - 1 : kTileWaves;
    int my_first = 0, my_count = 0;
    {
        const int base = ntile / nwork, rem = ntile % nwork;
        int first = 0;
        for (int w = 0; w < kTileWaves; ++w) {
            const int rank = nwork == kTileWaves ? w : (w == 3 ? 0 : (w < 3 ? w + 1 : w));
            const int cnt = w < nwork ? base + (rank < rem ? 1 : 0) : 0;
            if (w == wave) { my_first = first; my_count = cnt; }
            first += cnt;
        }
    }
    int my_I[kTilesPerWave], my_J[kTilesPerWave], my_q[kTilesPerWave];
#pragma unroll
    for (int sl = 0; sl < kTilesPerWave; ++sl) { my_I[sl] = -1; my_J[sl] = -1; my_q[sl] = -1; }
    {   // (my_q: the row of the tile's result, see 'part')
        int q = 0, row0 = 0;
        for (int Jb = jb0; Jb < jb1; ++Jb) {
            for (int I = tile_ilo(Jb, W); I <= Jb; ++I, ++q) {
                const int sl = q - my_first;
                if (sl >= 0 && sl < my_count) {
#pragma unroll
                    for (int u = 0; u < kTilesPerWave; ++u)
                        if (u == sl) { my_I[u] = I; my_J[u] = Jb; my_q[u] = row0 + I - tile_ilo(Jb, W); }
                }
            }
            row0 += (Jb - tile_ilo(Jb, W) + 1 + 7) & ~7;
        }
    }
    Tile t0, t1, t2;
    if (my_q[0] >= 0) load_scores(t0, links, my_I[0], my_J[0], lane, Lb, translen);
    if (my_q[1] >= 0) load_scores(t1, links, my_I[1], my_J[1], lane, Lb, translen);
    if (my_q[2] >= 0) load_scores(t2, links, my_I[2], my_J[2], lane, Lb, translen);

    const char *table_c = reinterpret_cast<const char *>(table);
    const char *match_c = reinterpret_cast<const char *>(match);
    auto cell = [&](int trow, int node) -> float * {
        return reinterpret_cast<float *>(const_cast<char *>(table_c) + (unsigned)(trow * L + node) * 4u);
    };
    const int ms1 = (int)a.ms1, ms2 = (int)a.ms2;   // the host checked that match indices fit 32 bits
    auto match_at = [&](int trow, int node) -> float {
        return to_float(*reinterpret_cast<const TM *>(match_c + (unsigned)(trow * ms1 + node * ms2) * (unsigned)sizeof(TM)));
    };

    // step 0: node 0 holds match[0][0] (even if that is -inf), everything else -inf
    const float m0 = match_at(0, 0);
    for (int q = tid; q < kMaxBlocksFast * kBlk; q += kTileWaves * kWave) {
        abuf[0][q / kBlk][q % kBlk] = q == 0 ? m0 : DAGX_NEG_INF;
        abuf[1][q / kBlk][q % kBlk] = DAGX_NEG_INF;
    }
    for (int q = tid; q < kPartRows * kBlk; q += kTileWaves * kWave) part[q / kBlk][q % kBlk] = DAGX_NEG_INF;
    for (int ob = wave; ob < nblk; ob += kTileWaves) {
        const int p = (jb0 + ob) * kBlk + lane;
        if (p < Lb) store_agent(cell(0, p), p == 0 ? m0 : DAGX_NEG_INF);
    }
    // ---- staging slots: match rows of own blocks wave and wave + 8, table
    //      rows of foreign blocks flo + wave and flo + wave + 8, all filled by the fetcher ----
    constexpr int kFetchSlots = 2;
    int f_blk[kFetchSlots];
#pragma unroll
    for (int u = 0; u < kFetchSlots; ++u) {   // dealt from the last wave down: the first waves are the ones that own blocks
        const int fb = flo + (kTileWaves - 1 - wave) + kTileWaves * u;
        f_blk[u] = fb < jb0 ? fb : -1;
    }
    const int *below = prog + (g > 0 ? g - 1 : 0);
    auto lds_addr = [&](const void *p) -> unsigned { return (unsigned)reinterpret_cast<uintptr_t>(p); };
    const bool fetcher = wave == kTileWaves - 1;
    int seen = 0;   // last progress value of the group below that the fetcher has read
    // The fetcher works one step ahead: in phase A of step s it waits for what it requested
    // a step ago (the rows phase B of step s reads), then requests the match rows of step s + 1, the foreign table
    // rows of step s + 1 if the snapshot of the producer's progress word (requested a step ago) shows them
    // published, and the next snapshot.  Only when the producer is less than two steps ahead does it poll the word
    // and fetch in the same step (one memory round trip inside phase A, which used to be every step's price).
    int rows_issued = 0;   // the foreign table rows of steps <= rows_issued have been requested
    auto issue_match = [&](const int s2, const int lane) __attribute__((always_inline)) {
        const int par = s2 & 1;
        const TM *mrow = reinterpret_cast<const TM *>(match_c + (unsigned)((s2 < mcap ? s2 : mcap) * ms1) * (unsigned)sizeof(TM));
        for (int ob = 0; ob < nblk; ++ob) {
            const int pm = (jb0 + ob) * kBlk + lane, pmc = pm < Lb ? pm : Lb - 1;
            dma_elem<TM>(lds_addr(&stage_m[par][ob & (kTileWaves - 1)][ob / kTileWaves][0]), mrow, (unsigned)(pmc * ms2) * (unsigned)sizeof(TM));
        }
    };
    auto issue_rows = [&](const int s2, const int lane) __attribute__((always_inline)) {
        const int par = s2 & 1;
        for (int fb = flo; fb < jb0; ++fb) {
            const int q = fb - flo, pf = fb * kBlk + lane, pfc = pf < Lb ? pf : Lb - 1;
            dma_dword_agent(lds_addr(&stage_f[par][kTileWaves - 1 - (q & (kTileWaves - 1))][q / kTileWaves][0]), table_c + (unsigned)(s2 * L) * 4u, (unsigned)pfc * 4u);
        }
        rows_issued = s2;
    };
    auto fetch_step = [&](const int s) __attribute__((always_inline)) {
        // (the fetcher's lane arithmetic is redone every step, on purpose: computed ahead of the loop over the steps it
        //  would hold registers that the tiles need)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        wait_vmem_all();   // everything requested a step ago
        if (consumer && s < Tb - 1) {
            const int snap = __builtin_amdgcn_readfirstlane(stage_p[s & 1][0]);
            if (snap > seen) seen = snap;
            if (rows_issued < s) {   // not requested yet: poll the producer's word
                int spins = 0;
                while (seen < s) {   // the rows of step s are published once the word reaches s
                    seen = __builtin_amdgcn_readfirstlane(load_agent(below));
                    if (seen >= s) break;
                    __builtin_amdgcn_s_sleep(2);
                    if (++spins > kSpinLimit) { s_abort = 1; break; }
                }
                if (seen >= s) { issue_rows(s, ln); wait_vmem_all(); }
            }
        }
        if (s + 1 < Tb) {
            issue_match(s + 1, ln);
            if (consumer && s + 1 < Tb - 1) {
                if (seen >= s + 1) issue_rows(s + 1, ln);
                dma_dword_agent(lds_addr(&stage_p[(s + 1) & 1][0]), below, 0u);
            }
        }
    };
    // The fetcher's instructions are what a step waits for where windows are long, and the wave that shares its SIMD multiplies tiles
    // meanwhile: without priority matrix instructions make it later than vector ones did, by up to 0.2 us a step.  Alignment, us, DPP sums /
    // matrix sums / those and the fetcher first: B = 1, L = 1024, T = 53 159.1 / 168.1 / 157.0, T = 14 74.1 / 77.2 / 72.8; B = 24, L = 960, T = 14
    // 78.2 / 82.5 / 78.3; B = 1, L = 640, T = 41 89.4 / 95.2 / 89.2; B = 64, L = 1024, T = 30 165.1 / 165.2 / 156.2; B = 64, L = 512, T = 29
    // 80.4 / 81.5 / 79.5; B = 1, L = 256, transitions of at most 64, T = 29 44.3 / 45.8 / 43.3; B = 130, L = 400, of at most 180, T = 41
    // 103.2 / 90.4 / 90.2.  (Priority only while it fetches: B = 24, L = 960, T = 14 80.5; B = 1, L = 1024, T = 20 89.1 for 86.3.)
    if (fetcher) __builtin_amdgcn_s_setprio(3);
    if (fetcher && Tb > 1) {   // what phase B of step 1 needs
        issue_match(1, lane);
        if (consumer && 1 < Tb - 1) dma_dword_agent(lds_addr(&stage_p[1][0]), below, 0u);
    }
    wait_vmem_all();
    __syncthreads();

    // What phase B needs for the block this wave owns (block jb0 + wave) does not change from step to step: its
    // first tile, its number of tiles and where its tile results lie.
    const bool own0 = wave < nblk;
    const int own_J = jb0 + wave, own_ilo = tile_ilo(own_J, W), own_nt = own_J - own_ilo + 1;
    auto part_row0 = [&](const int Jb) -> int {   // first result row of owned block Jb
        int row0 = 0;
        for (int J2 = jb0; J2 < Jb; ++J2) row0 += (J2 - tile_ilo(J2, W) + 1 + 7) & ~7;
        return row0;
    };
    const float *part_own = &part[own0 ? part_row0(own_J) : 0][lane];

    // the cell values of one owned block: maximum over its tiles (the first tile that attains it is remembered), plus
    // the match score; written to LDS for the next step and to the table
    auto finish_block = [&](const int Jb, const int ilo, const float best, const int from, const unsigned mraw, const int s, const int nxt,
                            const int lane) __attribute__((always_inline)) {
        const int p = Jb * kBlk + lane;
        const bool inband = p >= s && p <= slack + s;
        const float v = inband ? best + dma_decode<TM>(mraw) : DAGX_NEG_INF;   // second (and last) rounding of the cell
        abuf[nxt][Jb][lane] = v;
        if (p < Lb) { store_agent(cell(s, p), v); srcblk[s * spitch + p] = (unsigned char)(ilo + from); }
    };
    // maximum of eight tile results and the first place that holds it
    auto best_of_8 = [&](const float (&pv)[8], float &m, int &f) __attribute__((always_inline)) {
        m = max3(pv[0], pv[1], pv[2]);
        m = max3(m, pv[3], pv[4]);
        m = max3(m, pv[5], pv[6]);
        m = max3(m, pv[7], pv[7]);
        f = 7;
#pragma unroll
        for (int u = 6; u >= 0; --u) f = pv[u] == m ? u : f;
    };

    int cur = 0;
    for (int s = 1; s < Tb; ++s) {
        const int nxt = cur ^ 1;
        // ---- phase A: tile max-plus products; the fetcher's copies ----
        if (__builtin_expect(fetcher, 0)) fetch_step(s);
        {
            // The scores for a tile are requested one tile ahead of its arithmetic.  A tile whose predecessor block
            // holds no finite score, or whose block lies outside the band, is skipped.
            float av[kTilesPerWave];
            bool geo[kTilesPerWave];
#define DAGX_ALIGN_READ(SL)                                                                        \
            geo[SL] = my_q[SL] >= 0 && my_J[SL] * kBlk <= slack + s && my_J[SL] * kBlk + kBlk - 1 >= s; \
            if (geo[SL]) av[SL] = abuf[cur][my_I[SL]][lane];
#define DAGX_ALIGN_TILE(SL, TILE)                                                                  \
            if (my_q[SL] >= 0) {                                                                   \
                float best = DAGX_NEG_INF;                                                         \
                if (geo[SL] && __builtin_amdgcn_ballot_w64(av[SL] > DAGX_NEG_INF) != 0)           \
                    best = tile_maxplus(TILE, av[SL]);                                             \
                part[my_q[SL]][lane] = best;                                                       \
            }
            DAGX_ALIGN_READ(0)
            DAGX_ALIGN_READ(1)
            DAGX_ALIGN_TILE(0, t0)
            DAGX_ALIGN_READ(2)
            DAGX_ALIGN_TILE(1, t1)
            DAGX_ALIGN_TILE(2, t2)
#undef DAGX_ALIGN_READ
#undef DAGX_ALIGN_TILE
        }
        // This wave's stores of step s-1 were issued in that step's phase B, a whole phase A ago: waiting for them
        // here costs nothing, and behind the barrier every wave has done so -- the progress word can say s-1 at the
        // start of phase B already, not at the end of the step.  (The fetcher's stores: it waited at the top of its
        // fetch; its requests for step s+1 stay in flight until the top of its next fetch.)
        if (!fetcher) wait_vmem_all();
        __syncthreads();
        // ---- phase B ----
        if (__builtin_expect(tid == 0 && producer, 0)) store_agent(prog + g, s - 1);
        const int par = s & 1;
        const int gave_up_v = s_abort;   // set in phase A only; requested here, with the other LDS reads, and looked at behind the barrier
        if (own0) {
            const unsigned mraw = stage_m[par][wave][0][lane];
            float pv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) pv[u] = part_own[u * kBlk];
            float best; int from;
            best_of_8(pv, best, from);
            if (!(best > DAGX_NEG_INF)) from = 0;
            for (int u0 = 8; u0 < own_nt; u0 += 8) {   // more than eight tiles: L > 512 with long links
#pragma unroll
                for (int u = 0; u < 8; ++u) pv[u] = part_own[(u0 + u) * kBlk];
                float m; int f;
                best_of_8(pv, m, f);
                if (m > best) { best = m; from = u0 + f; }
            }
            finish_block(own_J, own_ilo, best, from, mraw, s, nxt, lane);
        }
        for (int ob = wave + kTileWaves; ob < nblk; ob += kTileWaves) {   // a second owned block (narrow bands only)
            // (rare, so written to need few registers rather than to be fast: one tile result at a time,
            // and nothing of it computed ahead of the loop over the steps, where it would hold registers: hence 'ln')
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int Jb = jb0 + ob, ilo = tile_ilo(Jb, W), nt = Jb - ilo + 1;
            const float *pr = &part[part_row0(Jb)][ln];
            const unsigned mraw = stage_m[par][wave][ob / kTileWaves][ln];
            float best = DAGX_NEG_INF;
            int from = 0;   // first tile (= lowest predecessor block) that attains the maximum
            for (int u = 0; u < nt; ++u) {
                const float x = pr[u * kBlk];
                if (x > best) { best = x; from = u; }
            }
            finish_block(Jb, ilo, best, from, mraw, s, nxt, ln);
        }
        if (consumer && s < Tb - 1) {
#pragma unroll
            for (int u = 0; u < kFetchSlots; ++u) {
                if (f_blk[u] < 0) continue;
                abuf[nxt][f_blk[u]][lane] = f_blk[u] * kBlk + lane < Lb ? stage_f[par][wave][u][lane] : DAGX_NEG_INF;
            }
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(gave_up_v)) {
            if (tid == 0) { a.flags[b] = 1; store_agent(prog + g, 1 << 30); }
            return;
        }
        cur = nxt;
    }
    if (producer) {
        wait_vmem_all();
        __syncthreads();
        if (tid == 0) store_agent(prog + g, Tb - 1);
    }
}

// Walking the path backwards through the score table.  The sweep has recorded, for every cell, the lowest block of 64
// nodes that holds a best predecessor, so a step scans 64 candidates (lanes <-> nodes of that block): it re-evaluates
// fl32(A[t-1][i] + E[i][j]) -- the very operation of the sweep, hence bit-identical -- takes the maximum and, among the
// lanes that hold it, the lowest node: the first-index rule of torch.max (fs_plugins/custom_ops/dag_loss.py:253-257, :350).
//
// The steps are a serial chain, one wave per sample, so what bounds the walk is the latency of a step.  Read from memory a
// step's scores and transitions cost a round trip to HBM (0.61 us a step).  A path moves on by a few nodes a step, so it
// stays in a block of 64 nodes for several steps and nearly always finds its predecessor in that block or the one below:
// while wave 0 walks through block J out of LDS, the other waves bring in what a walk through block J - 1 reads (the
// transitions from its two predecessor blocks, and kWalkRows rows of their scores and of the source blocks, whichever
// step the walk enters with).  A predecessor further away is read from memory, a walk that leaves the staged rows or jumps
// over a block stages again in front of the next step.  Measured: see launch_align; when it does not pay: see walk_back.
constexpr int kWalkRows = 48;             // two buffers and the decoder's own 25 KB fit the 160 KB of a CU
constexpr int kWalkPitch = kBlk + 1;      // the lanes read a column of the transitions: no two in one bank
struct alignas(16) WalkStage {
    float e[2 * kBlk * kWalkPitch];       // E[(J-1)*64 + r][J*64 + c] at r * kWalkPitch + c, -inf where there is none
    float a[kWalkRows * 2 * kBlk];        // row r: A[hi - 1 - r] of blocks J - 1 and J
    unsigned src[kWalkRows * kBlk / 4];   // row r: source blocks of (hi - r, block J), a byte each
};
constexpr size_t kWalkLds = 2 * sizeof(WalkStage);

// Four neighbouring elements a lane: a CU takes one vector-memory instruction per 26 cycles whatever its width, and with one element
// a lane a block was 255 of them; now it is 90.  (Backtrack at B=64 L=512 T=64 24 -> 22.4 us, with the walker's priority; at
// B=16 L=1024 T=256, where a block of nodes is sixteen steps, the steps bound it: 65 us before and after.)
template <typename TL, int NT>
__device__ __forceinline__ void stage_walk(WalkStage &w, const float *A, const unsigned char *srcblk, int spitch, const TL *links,
                                           int L, int translen, int J, int hi) {
    constexpr int kHelpers = NT - kWave, kQuads = kBlk / 4;
    const int q = (int)threadIdx.x - kWave;
    typedef typename Quad<TL>::V V;
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    constexpr int kEQuads = 2 * kBlk * kQuads, kAQuads = kWalkRows * 2 * kQuads, kSQuads = kWalkRows * kBlk / 16;
    constexpr int kE = (kEQuads + kHelpers - 1) / kHelpers, kA = (kAQuads + kHelpers - 1) / kHelpers;
    static_assert(kSQuads <= kHelpers, "one load of source blocks a thread");
    V ve[kE];
    f32x4 va[kA];
    u32x4 vs;
    const int64_t most = (int64_t)L * translen - 4;   // (walk_back: at least 0)
    // element k of quad u is at place at_e[u] + k of the sample's links, its distance is d_e[u] + k; it is one for k < end_e[u]
    int64_t at_e[kE];
    int d_e[kE], end_e[kE];
#pragma unroll
    for (int u = 0; u < kE; ++u) {   // everything is requested before anything is stored
        const int x = q + u * kHelpers, i = (J - 1) * kBlk + x / kQuads, j = J * kBlk + 4 * (x % kQuads);
        d_e[u] = j - i - 1;
        at_e[u] = (int64_t)i * translen + d_e[u];
        end_e[u] = i >= 0 && x < kEQuads ? min(L - j, translen - d_e[u]) : 0;
        // (a load that would leave the sample is moved inside; its elements, at an end of the sample, are read one by one below)
        const int64_t at = at_e[u] < 0 ? 0 : at_e[u] > most ? most : at_e[u];
        __builtin_memcpy(&ve[u], links + at, sizeof(V));
    }
#pragma unroll
    for (int u = 0; u < kA; ++u) {   // (up to three elements past a row's end: row + 1 <= hi is a row of the table)
        const int x = q + u * kHelpers, row = hi - 1 - x / (2 * kQuads), i = (J - 1) * kBlk + 4 * (x % (2 * kQuads));
        __builtin_memcpy(&va[u], A + (row >= 0 && i >= 0 && i < L && x < kAQuads ? (int64_t)row * L + i : 0), sizeof(f32x4));
    }
    {
        const int row = hi - q / (kBlk / 16), at = J * kBlk + 16 * (q % (kBlk / 16));   // (rows are padded to 16 bytes)
        vs = *reinterpret_cast<const u32x4 *>(srcblk + (q < kSQuads && row >= 1 && at < spitch ? (int64_t)row * spitch + at : 0));
    }
#pragma unroll
    for (int u = 0; u < kE; ++u) {
        const int x = q + u * kHelpers;
        if (x >= kEQuads) continue;
        float *const to = &w.e[(x / kQuads) * kWalkPitch + 4 * (x % kQuads)];
        if (__builtin_expect(at_e[u] >= 0 && at_e[u] <= most, 1)) {
#pragma unroll
            for (int k = 0; k < 4; ++k) to[k] = d_e[u] + k >= 0 && k < end_e[u] ? Quad<TL>::get(ve[u], k) : DAGX_NEG_INF;
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) to[k] = d_e[u] + k >= 0 && k < end_e[u] ? to_float(links[at_e[u] + k]) : DAGX_NEG_INF;
        }
    }
#pragma unroll
    for (int u = 0; u < kA; ++u) { const int x = q + u * kHelpers; if (x < kAQuads) *reinterpret_cast<f32x4 *>(&w.a[4 * x]) = va[u]; }
    if (q < kSQuads) *reinterpret_cast<u32x4 *>(&w.src[4 * q]) = vs;
}

// The walk with every step read from memory, by one wave, without LDS: the row of source blocks of the next step is fetched
// together with the candidates of this one (it does not depend on where the path goes), so a step costs one round trip.
// Arguments as walk_back_staged's.
template <typename TL, bool ZERO_FOR_DEAD, typename PUT>
__device__ __forceinline__ void walk_back_in_memory(const float *A, const unsigned char *srcblk, int spitch, const TL *links, int L,
                                                    int translen, int s, int j, int stop, PUT put) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & (kWave - 1);
    auto load_row = [&](int t) {   // L <= 1024 bytes: lane l holds bytes 16 l .. 16 l + 15 (rows are padded to 16 bytes)
        return *reinterpret_cast<const u32x4 *>(srcblk + (int64_t)t * spitch + (16 * lane < spitch ? 16 * lane : 0));
    };
    u32x4 row = {};
    if (s > stop) row = load_row(s);
    for (; s > stop; --s) {
        const int q = (j >> 2) & 3;
        const unsigned w = q == 0 ? row.x : q == 1 ? row.y : q == 2 ? row.z : row.w;
        const int I = (int)((unsigned)__builtin_amdgcn_readlane((int)w, j >> 4) >> (8 * (j & 3))) & 0xff;
        const int i = I * kBlk + lane, d = j - i - 1;
        const bool valid = d >= 0 && d < translen && i < L;
        const float e = to_float(links[valid ? (int64_t)i * translen + d : 0]);
        const float av = A[(int64_t)(s - 1) * L + (i < L ? i : L - 1)];
        if (s - 1 > stop) row = load_row(s - 1);
        const float x = valid ? av + e : DAGX_NEG_INF;
        const float top = wave64_max(x);
        j = I * kBlk + (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(x == top));   // the lowest lane among those that hold the maximum
        if (__builtin_expect(!(top > DAGX_NEG_INF), 0)) {
            if (!ZERO_FOR_DEAD) return;
            j = 0;
        }
        if (lane == 0) put(s - 1, j);
    }
}

// From cell (s, j) down to row `stop` by the whole workgroup: put(row, node), called by single lanes of wave 0, takes the
// predecessors found.  Where no candidate has a finite score the walk ends, or with ZERO_FOR_DEAD goes on from node 0.
// lds: kWalkLds bytes.  s, j are uniform over the workgroup.
// A step is a chain of dependent instructions of one wave, so its length is what counts: the byte that names the block and
// the scores and transitions of both blocks are read in one LDS round trip, in whose shade what is not part of the chain is
// done, and the nodes found are kept in a register, one a lane, and put 64 rows at a time.  While the path stays in the block
// a step has one jump, whose condition also covers what ends the run of steps (another block, a cell without a finite score):
// a step into a block further away has then been taken from the two at hand, and is taken again from memory.  Kernel, us, against
// a step with a jump for each of these and the keeping at its end: alignment B = 64, L = 512, T = 64 22.3 -> 18.7, B = 16, L = 1024,
// T = 256 64.1 -> 54.1 (0.21 us a step).
template <typename TL, int NT, bool ZERO_FOR_DEAD, typename PUT>
__device__ __forceinline__ void walk_back_staged(const float *A, const unsigned char *srcblk, int spitch, const TL *links, int L,
                                          int translen, int s, int j, int stop, WalkStage *lds, PUT put) {
    __shared__ int at[2][2];
    if (s <= stop) return;
    const bool walker = threadIdx.x < kWave;
    const int lane = threadIdx.x & (kWave - 1);
    int cur = 0, J = j / kBlk, hi = s;
    int mine = -1;   // the node found for the row whose number ends in `lane`
    if (!walker) stage_walk<TL, NT>(lds[0], A, srcblk, spitch, links, L, translen, J, hi);
    __syncthreads();
    for (int round = 0;; ++round) {
        const int next_hi = s - 1;
        if (!walker) {
            if (J > 0 && next_hi > stop) stage_walk<TL, NT>(lds[cur ^ 1], A, srcblk, spitch, links, L, translen, J - 1, next_hi);
        } else {
            __builtin_amdgcn_s_setprio(3);   // (three of the other waves share its SIMD)
            const WalkStage &w = lds[cur];
            const unsigned char *src = reinterpret_cast<const unsigned char *>(w.src) + (hi - s) * kBlk;
            const float *arow = w.a + (hi - s) * 2 * kBlk + lane, *ecol = w.e + lane * kWalkPitch;
            while (s > stop && hi - s < kWalkRows && j >> 6 == J) {   // (-1: no block)
                // as far as rows are staged and nodes found can be kept, while the path stays in the block
                const int until = max(max(stop, hi - kWalkRows), (s - 1) & ~(kWave - 1));
                int c = j & (kBlk - 1), from, byte, last = -1;     // last: where a step's node is to be kept, behind the next one's reads
                float x, top;
                unsigned long long stays;
                do {
                    from = c;
                    byte = src[c];
                    float e0 = ecol[c], e1 = ecol[kBlk * kWalkPitch + c], a0 = arow[0], a1 = arow[kBlk];
                    __builtin_amdgcn_sched_barrier(0);
                    mine = lane == last ? J * kBlk + c : mine;
                    --s;
                    last = s & (kWave - 1);
                    src += kBlk; arow += 2 * kBlk;
                    const bool more = s > until;
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("" : "+v"(byte), "+v"(e0), "+v"(e1), "+v"(a0), "+v"(a1));   // (else read one after the other)
                    x = byte == J ? a1 + e1 : a0 + e0;
                    stays = __builtin_amdgcn_ballot_w64(byte == J);
                    top = wave64_max(x);
                    // lowest lane among those that hold the maximum
                    const unsigned long long at_top = __builtin_amdgcn_ballot_w64(x == top);
                    c = (int)__builtin_ctzll(at_top);
                    stays &= at_top & __builtin_amdgcn_ballot_w64(top > DAGX_NEG_INF);   // (no lane: a NaN)
                    if (!more) break;
                } while (stays != 0);
                const int I = __builtin_amdgcn_readfirstlane(byte);
                if (__builtin_expect((unsigned)(J - I) > 1u, 0)) {
                    const int i = I * kBlk + lane, d = J * kBlk + from - i - 1;
                    const bool valid = d >= 0 && d < translen && i < L;
                    const float e = to_float(links[valid ? (int64_t)i * translen + d : 0]);
                    const float av = A[(int64_t)s * L + (i < L ? i : L - 1)];
                    x = valid ? av + e : DAGX_NEG_INF;
                    top = wave64_max(x);
                    c = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(x == top));
                }
                j = __builtin_amdgcn_readfirstlane(top > DAGX_NEG_INF ? I * kBlk + c : ZERO_FOR_DEAD ? 0 : -1);
                mine = lane == last ? j : mine;
                if (last == 0) {
                    if (mine >= 0) put(s + lane, mine);
                    mine = -1;
                }
            }
            if (lane == 0) { at[round & 1][0] = s; at[round & 1][1] = j; }
        }
        __syncthreads();
        s = __builtin_amdgcn_readfirstlane(at[round & 1][0]);
        j = __builtin_amdgcn_readfirstlane(at[round & 1][1]);
        if (s <= stop || j < 0) {
            if (walker && mine >= 0) put((s & ~(kWave - 1)) + lane, mine);
            return;
        }
        cur ^= 1;
        if (j / kBlk == J - 1 && next_hi > stop && next_hi >= s && next_hi - s < kWalkRows) {
            J -= 1; hi = next_hi;
        } else {
            J = j / kBlk; hi = s;
            if (!walker) stage_walk<TL, NT>(lds[cur], A, srcblk, spitch, links, L, translen, J, hi);
            __syncthreads();
        }
    }
}

// STAGED: lds holds kWalkLds bytes.  A path with few steps a block, as Viterbi decoding finds where no transition stands out,
// walks in memory all the same: a block staged cost as much as about four steps from memory (2.3 and 0.6 us, with one element a load; Viterbi decoding
// at B=64, paths of 13 nodes: L=512 staged 229 us, in memory 221; L=1024 982 and 967).
constexpr int kWalkStepsPerBlock = 4;
template <typename TL, int NT, bool ZERO_FOR_DEAD, bool STAGED, typename PUT>
__device__ __forceinline__ void walk_back(const float *A, const unsigned char *srcblk, int spitch, const TL *links, int L,
                                          int translen, int s, int j, int stop, WalkStage *lds, PUT put) {
    if (STAGED && L >= 4 && s - stop >= kWalkStepsPerBlock * (j / kBlk + 1))   // (four elements a load)
        walk_back_staged<TL, NT, ZERO_FOR_DEAD>(A, srcblk, spitch, links, L, translen, s, j, stop, lds, put);
    else if (threadIdx.x < kWave)
        walk_back_in_memory<TL, ZERO_FOR_DEAD>(A, srcblk, spitch, links, L, translen, s, j, stop, put);
}

// The backtrack of the alignment, one workgroup per sample.  A sample that the pipeline gave up on (flags[b] set) is
// done again here, from scratch, by the one-workgroup method.  (A launch of its own for the flagged samples, which are rare, would cost every call its latency.)
constexpr int kOneGroupThreads = 1024;
template <typename TM, typename TL, bool TRACE_LDS, bool STAGED>
__global__ __launch_bounds__(kOneGroupThreads) void dag_backtrack_kernel(
    const float *__restrict__ table, const unsigned char *__restrict__ srcblk_all, const int *__restrict__ flags, AlignArgs a) {
    extern __shared__ __align__(16) float lds_a[];
    const int b = blockIdx.x;
    if (flags[b]) {
        align_one_sample<TM, TL, kOneGroupThreads, TRACE_LDS>(a, b, lds_a);
        return;
    }
    const int T = a.T, L = a.L, translen = a.translen;
    int64_t *path = a.path + (int64_t)b * L;
    if (threadIdx.x < kWave)
        for (int j = threadIdx.x; j < L; j += kWave) path[j] = -1;
    const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
    if (!(Tb >= 1 && Lb >= 1 && Tb <= T && Lb <= L && Tb <= Lb)) return;
    const float *A = table + (int64_t)b * T * L;
    const int spitch = srcblk_pitch(L);
    if (!(A[(int64_t)(Tb - 1) * L + Lb - 1] > DAGX_NEG_INF)) return;   // no finite path
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");     // the -1 fill precedes the path entries (same wave)
    if (threadIdx.x == 0) path[Lb - 1] = Tb - 1;
    walk_back<TL, kOneGroupThreads, false, STAGED>(A, srcblk_all + (int64_t)b * T * spitch, spitch, static_cast<const TL *>(a.links) + (int64_t)b * L * translen,
                                           L, translen, Tb - 1, Lb - 1, 0, reinterpret_cast<WalkStage *>(lds_a),
                                           [&](int t, int j) { path[j] = t; });   // (the walk does not end early on a finite path)
}

constexpr size_t kAlignLdsBudget = 144 * 1024;
// A walk that stages takes the LDS of a CU, so batches beyond the 256 CUs go in turns; walks in memory share a CU.  The
// alignment's staged walk is short enough for two turns of graphs of more than two blocks (backtrack, us, in memory / staged:
// B=300 L=64 T=16 12.9 / 14.2, L=184 T=32 25.6 / 23.2, L=512 T=64 50 / 43; B=512 L=184 25.5 / 24.5, L=328 T=41 32.9 / 34.9;
// B=1024 L=64 15.4 / 28.0, L=100 T=24 21.6 / 37.8); the decoder's select kernel is not (B=300 L=184, 46 steps, paths of 27
// nodes: 23.7 / 26.7; L=64, 16 steps, paths of 7: 12.0 / 15.4).
static bool staged_alignment(int B, int L) { return B <= 256 || (B <= 512 && L > 2 * kBlk); }
static bool staged_decode(int B) { return B <= 256; }

static bool trace_fits_lds(int T, int L) {
    return L <= 65535 && (size_t)L * 8 + (size_t)T * L * 2 <= kAlignLdsBudget;
}

// workspace: [score table B*T*L f32 | sync 16 + B*C ints | flags B ints | source blocks B*T*L bytes] (tile path) then
//            [trace B*T*L i32] when the back-pointers of the one-workgroup kernel do not fit LDS
static size_t align_tile_words(int B, int T, int L, int translen) {
    const int C = align_groups(B, T, L, translen);
    // the last terms: one byte per cell in rows of srcblk_pitch(L) bytes, and room to start them on a 16-byte boundary
    return C > 0 ? (size_t)B * T * L + 16 + (size_t)B * C + (size_t)B + 4 + (size_t)B * T * srcblk_pitch(L) / 4 : 0;
}
size_t align_workspace_bytes(int B, int T, int L, int translen) {
    return align_tile_words(B, T, L, translen) * 4 + (trace_fits_lds(T, L) ? 0 : (size_t)B * T * L * sizeof(int32_t));
}

// the pipeline words cleared; the flags of the samples ('nflags' words behind them) cleared too, or set (a test switch)
__global__ void dag_align_fill_kernel(int *p, int n, int nflags, int flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i >= n - nflags ? flag : 0;
}

// Dynamic LDS beyond the default limit: raised once per device and instantiation (bit d of `done`: device d), to the most
// any launch asks for.
static int raise_lds_limit(const void *kern, size_t bytes, std::atomic<unsigned long long> &done, const char *who) {
    int device = 0;
    (void)hipGetDevice(&device);
    const unsigned long long bit = 1ull << (device & 63);
    if (done.load(std::memory_order_acquire) & bit) return DAGX_OK;
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) { set_error("%s: cannot reserve %zu bytes of LDS: %s", who, bytes, hipGetErrorString(e)); return DAGX_ERR_LAUNCH; }
    done.fetch_or(bit, std::memory_order_release);
    return DAGX_OK;
}
template <typename TM, typename TL, int SPACING>
static int prepare_align_chunks() {
    static std::atomic<unsigned long long> done{0};
    return raise_lds_limit(reinterpret_cast<const void *>(dag_align_chunks_kernel<TM, TL, SPACING>), kChunkLdsBytes, done, "dag_best_alignment");
}
template <typename TM, typename TL, int SPACING>
static int launch_align_chunks(AlignTileArgs &ta, const char *who, hipStream_t st) {
    ta.plan = chunk_plan<SPACING>(ta.translen, ta.C, align_costs<SPACING>(ta.translen));
    if (int rc = prepare_align_chunks<TM, TL, SPACING>()) return rc;
    hipLaunchKernelGGL((dag_align_chunks_kernel<TM, TL, SPACING>), dim3(((ta.B + 7) & ~7) * ta.C), dim3(kTileWaves * kWave), kChunkLdsBytes, st, ta);
    return check_launch(who);
}
template <typename TM, typename TL>
static int launch_align_sweep(AlignTileArgs &ta, const char *who, hipStream_t st) {
    const int NB = (ta.L + kBlk - 1) / kBlk;
    if (!align_in_chunks(ta.B, ta.T, ta.L, ta.translen)) {
        const int W = (ta.translen + kBlk - 1) / kBlk;
        int first[kTileCap + 2];
        for (int nb = 0; nb <= kMaxBlocksFast; ++nb) {
            partition_blocks(nb, W, ta.C, first);
            for (int q = 0; q <= ta.C && q < 12; ++q) ta.plan.gtab[0][nb][q] = (unsigned char)first[q];
        }
        hipLaunchKernelGGL((dag_align_steps_kernel<TM, TL>), dim3(((ta.B + 7) & ~7) * ta.C), dim3(kTileWaves * kWave), 0, st, ta);
        return check_launch(who);
    }
    return align_spacing(NB, ta.C) == 2 ? launch_align_chunks<TM, TL, 2>(ta, who, st) : launch_align_chunks<TM, TL, 1>(ta, who, st);
}
constexpr size_t kBacktrackMostLds = kAlignLdsBudget > kWalkLds ? kAlignLdsBudget : kWalkLds;   // (the redo alone asks for at most the former)
template <typename TM, typename TL, bool TRACE_LDS, bool STAGED>
static int prepare_backtrack() {
    static std::atomic<unsigned long long> done{0};
    return raise_lds_limit(reinterpret_cast<const void *>(dag_backtrack_kernel<TM, TL, TRACE_LDS, STAGED>), kBacktrackMostLds, done, "dag_best_alignment");
}

template <typename TM, typename TL>
static int prepare_backtracks() {
    int rc = prepare_backtrack<TM, TL, true, true>();
    if (!rc) rc = prepare_backtrack<TM, TL, true, false>();
    if (!rc) rc = prepare_backtrack<TM, TL, false, true>();
    return rc ? rc : prepare_backtrack<TM, TL, false, false>();
}

template <typename TM, typename TL>
static int launch_align(AlignArgs a, void *workspace, hipStream_t st) {
    constexpr int NT = 1024;
    const size_t tile_words = align_tile_words(a.B, a.T, a.L, a.translen);
    a.trace_ws = reinterpret_cast<int32_t *>(static_cast<float *>(workspace) + tile_words);
    int C = align_groups(a.B, a.T, a.L, a.translen);
    const int64_t span = (int64_t)(a.T - 1) * (a.ms1 < 0 ? -a.ms1 : a.ms1) + (int64_t)(a.L - 1) * (a.ms2 < 0 ? -a.ms2 : a.ms2);
    if (span >= (1LL << 31) / (int64_t)sizeof(TM) || a.ms1 < 0 || a.ms2 < 0 || force_log_domain()) C = 0;
    if (C > 0) {
        AlignTileArgs ta{};
        ta.match = a.match; ta.ms0 = a.ms0; ta.ms1 = a.ms1; ta.ms2 = a.ms2; ta.links = a.links;
        ta.out_len = a.out_len; ta.tgt_len = a.tgt_len; ta.B = a.B; ta.T = a.T; ta.L = a.L; ta.translen = a.translen;
        ta.table = static_cast<float *>(workspace);
        ta.sync = reinterpret_cast<int *>(ta.table + (size_t)a.B * a.T * a.L);
        ta.flags = ta.sync + 16 + a.B * C;
        ta.srcblk = reinterpret_cast<unsigned char *>((reinterpret_cast<uintptr_t>(ta.flags + a.B) + 15) & ~(uintptr_t)15);
        ta.C = C; ta.mcap = a.T - 1; ta.decode = 0;
        const int nfill = 16 + a.B * C + a.B;
        hipLaunchKernelGGL(dag_align_fill_kernel, dim3((nfill + 255) / 256), dim3(256), 0, st, ta.sync, nfill, a.B, redo_every_sample() ? 1 : 0);
        int rc = check_launch("dag_align_fill");
        if (rc) return rc;
        if ((rc = launch_align_sweep<TM, TL>(ta, "dag_align_sweep", st))) return rc;
        // the backtrack, and the samples that the pipeline gave up on.  (float32, kernel time: walked in memory 39.5 us at
        // B=64 L=512 T=64 and 172 us at B=16 L=1024 T=256, out of LDS 18.7 and 54 us.)
        const bool in_lds = trace_fits_lds(a.T, a.L);
        const size_t redo_lds = (size_t)a.L * 8 + (in_lds ? (size_t)a.T * a.L * 2 : (size_t)0);
        const bool staged = staged_alignment(a.B, a.L);
        const size_t lds = staged && redo_lds < kWalkLds ? kWalkLds : redo_lds;
        auto kern = in_lds ? (staged ? dag_backtrack_kernel<TM, TL, true, true> : dag_backtrack_kernel<TM, TL, true, false>)
                           : (staged ? dag_backtrack_kernel<TM, TL, false, true> : dag_backtrack_kernel<TM, TL, false, false>);
        if ((rc = prepare_backtracks<TM, TL>())) return rc;
        hipLaunchKernelGGL(kern, dim3(a.B), dim3(kOneGroupThreads), lds, st, ta.table, ta.srcblk, ta.flags, a);
        return check_launch("dag_backtrack");
    }
    if (trace_fits_lds(a.T, a.L)) {
        size_t lds = (size_t)a.L * 8 + (size_t)a.T * a.L * 2;
        auto kern = dag_align_kernel<TM, TL, NT, true>;
        if (lds > 48 * 1024) {
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) { set_error("dag_best_alignment: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e)); return DAGX_ERR_LAUNCH; }
        }
        hipLaunchKernelGGL(kern, dim3(a.B), dim3(NT), lds, st, a);
    } else {
        hipLaunchKernelGGL((dag_align_kernel<TM, TL, NT, false>), dim3(a.B), dim3(NT), (size_t)a.L * 8, st, a);
    }
    return check_launch("dag_align");
}

template <typename TM>
static int dispatch_align(int ldt, const AlignArgs &a, void *ws, hipStream_t st) {
    switch (ldt) {
        case DAGX_F32: return launch_align<TM, float>(a, ws, st);
        case DAGX_F16: return launch_align<TM, __half>(a, ws, st);
        default: return launch_align<TM, bf16_t>(a, ws, st);
    }
}

// ================================================================================================
// Viterbi decoding (fs_plugins/models/glat_decomposed_with_link.py:720-777)
// ================================================================================================
// The decoder's recursion  reach_t[j] = max_i fl32(reach_{t-1}[i] + E[i][j]) (+ u[j] in the joint
// form),  reach_0[j] = E[0][j] (+ u[0]) + u[j],  is the alignment sweep above with the table row
// s = t + 1, node 0 alone in row 0, and a three-row "match": row 0 = (u[0] or 0 at node 0), row 1 = u,
// rows >= 2 = (u or 0).  Every sample runs all `steps` = max_length + 1 rows and nothing is pruned
// towards the end, because a path may stop after any step: its score is reach_t[j] + E[j][L_b-1],
// divided by (t+1)^beta.  The sweep leaves the score table and the source blocks; one workgroup per
// sample then finds the best (t, j), walks back and collapses the tokens.
constexpr int kDecodeMaxSteps = 2049;   // max_length <= 2048 (= 2 L at L = 1024)
constexpr int kDecodeThreads = 1024;

// sync words <- 0, flags <- `flag`, match rows of every sample
__global__ void viterbi_prep_kernel(int *sync, int nsync, int *flags, int flag, const float *__restrict__ node_logp,
                                    int B, int L, int joint, float *__restrict__ match3) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nsync) sync[i] = 0;
    if (i < B) flags[i] = flag;
    if (i < B * L) {
        const int b = i / L, j = i - b * L;
        const float u = node_logp[i];
        float *m = match3 + (int64_t)b * 3 * L;
        m[j] = (joint && j == 0) ? u : 0.0f;
        m[L + j] = u;
        m[2 * L + j] = joint ? u : 0.0f;
    }
}

// The table and the source blocks of one sample by one workgroup (a team of lanes <-> node, every lane scanning
// its predecessors in ascending order with a strict '>'): for the samples the pipeline did not do.
template <typename TL, int NT>
__global__ __launch_bounds__(NT) void viterbi_table_kernel(
    const float *__restrict__ match3, const TL *__restrict__ links_all, const int64_t *__restrict__ out_len,
    const int *__restrict__ flags, int T, int L, int translen, float *__restrict__ table_all,
    unsigned char *__restrict__ srcblk_all) {
    extern __shared__ float lds_v[];   // 2 L floats
    const int b = blockIdx.x, tid = threadIdx.x;
    if (!flags[b]) return;
    const int Lb = (int)out_len[b];
    if (!(Lb >= 1 && Lb <= L)) return;
    const float *m = match3 + (int64_t)b * 3 * L;
    const TL *links = links_all + (int64_t)b * L * translen;
    float *table = table_all + (int64_t)b * T * L;
    const int spitch = srcblk_pitch(L);
    unsigned char *srcblk = srcblk_all + (int64_t)b * T * spitch;
    float *fprev = lds_v, *fcur = lds_v + L;
    for (int j = tid; j < L; j += NT) {
        const float v = j == 0 ? m[0] : DAGX_NEG_INF;
        fprev[j] = v;
        if (j < Lb) table[j] = v;
    }
    __syncthreads();
    // a team of kTeam lanes <-> node, as in align_one_sample
    constexpr int kTeam = 8, R = 8;
    const int team = tid / kTeam, sub = tid % kTeam;
    const unsigned rs = (unsigned)(translen - 1);   // E[i][j-i-1] sits at links[i*(translen-1) + j-1]: 32-bit offsets
    for (int s = 1; s < T; ++s) {
        const float *mrow = m + (s < 2 ? s : 2) * L;
        for (int j = tid; j < Lb && j < s; j += NT) {   // not reachable in s steps
            fcur[j] = DAGX_NEG_INF;
            table[(int64_t)s * L + j] = DAGX_NEG_INF;
            srcblk[s * spitch + j] = 0;
        }
        for (int j = s + team; j < Lb; j += NT / kTeam) {
            const float mj = mrow[j];
            int ilo = j - translen; if (ilo < s - 1) ilo = s - 1;
            float best = DAGX_NEG_INF;
            int arg = ilo;
            const unsigned o_last = (unsigned)(j - 1) * (unsigned)translen;   // the offset of i = j-1, the largest
            unsigned o = (unsigned)(ilo + sub) * rs + (unsigned)(j - 1);
            for (int i0 = ilo + sub; i0 < j; i0 += kTeam * R, o += kTeam * R * rs) {
                float e[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const unsigned oc = o + (unsigned)(r * kTeam) * rs;
                    e[r] = to_float(links[oc < o_last ? oc : o_last]);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int i = i0 + r * kTeam;
                    const float x = i < j ? fprev[i < j ? i : j - 1] + e[r] : DAGX_NEG_INF;
                    if (x > best) { best = x; arg = i; }
                }
            }
#pragma unroll
            for (int w = kTeam / 2; w > 0; w >>= 1) {
                const float bo = __shfl_xor(best, w, kWave);
                const int ao = __shfl_xor(arg, w, kWave);
                if (bo > best || (bo == best && ao < arg)) { best = bo; arg = ao; }
            }
            if (sub == 0) {
                const float val = best + mj;
                fcur[j] = val;
                table[(int64_t)s * L + j] = val;
                srcblk[s * spitch + j] = (unsigned char)(arg / kBlk);
            }
        }
        __syncthreads();
        float *sw = fprev; fprev = fcur; fcur = sw;
    }
}

// the lowest index among the lanes whose value equals the wave's maximum; `top` receives that maximum
__device__ __forceinline__ int wave_first_argmax(float v, int idx, float &top) {
    top = wave64_max(v);
    const float cand = v == top ? (float)idx : 3.0e7f;   // indices < 2^24 are exact in float
    return (int)-wave64_max(-cand);
}

struct DecodeArgs {
    const float *table; const unsigned char *srcblk; const void *links;
    const int64_t *out_len, *node_tokens;
    const float *penalty;
    int T, L, translen, max_length;
    int64_t pad;
    int64_t *out_tokens, *out_count, *pred_length, *nodes;
};

// One workgroup per sample: the best node of every step, the best length, the walk back (walk_back) and the tokens.
template <typename TL, bool STAGED>
__global__ __launch_bounds__(kDecodeThreads) void viterbi_select_kernel(DecodeArgs a) {
    extern __shared__ __align__(16) float lds_walk[];
    __shared__ int s_star;
    __shared__ float sbest[kDecodeMaxSteps];
    __shared__ int sidx[kDecodeMaxSteps];
    __shared__ int walk[kDecodeMaxSteps];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int L = a.L, T = a.T, translen = a.translen, n_max = a.max_length;
    const int Lb = (int)a.out_len[b];
    const float *A = a.table + (int64_t)b * T * L;
    const int spitch = srcblk_pitch(L);
    const unsigned char *srcblk = a.srcblk + (int64_t)b * T * spitch;
    const TL *links = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    const int64_t *tok = a.node_tokens + (int64_t)b * L;
    int64_t *out_tokens = a.out_tokens + (int64_t)b * n_max;
    int64_t *nodes = a.nodes + (int64_t)b * n_max;
    const bool sane = Lb >= 1 && Lb <= L;

    // transition of every node to the last one: lane l holds nodes l, l + 64, ...
    float to_end[kMaxBlocksFast];
#pragma unroll
    for (int c = 0; c < kMaxBlocksFast; ++c) {
        const int j = c * kWave + lane, d = Lb - 1 - j - 1;
        const bool ok = sane && j < Lb && d >= 0 && d < translen;
        to_end[c] = ok ? to_float(links[(int64_t)j * translen + d]) : DAGX_NEG_INF;
    }
    // best node of every step (first index among equals, over all L nodes as the tensor formulation);
    // a wave takes kRows steps at a time, kCols blocks of 64 nodes of each, so that it waits for sixteen loads at once
    constexpr int kRows = 4, kCols = 4, kWaves = kDecodeThreads / kWave;
    const int nblk = (L + kWave - 1) / kWave;
    const unsigned in_last = min(lane, L - 1 - (nblk - 1) * kWave);
    for (int t0 = wave * kRows; t0 < n_max; t0 += kWaves * kRows) {
        // An address is a scalar part and one of two offsets a lane, formed when it is needed: kept from one turn to the next,
        // sixteen of them a lane took the kernel to 128 registers and scratch, and so to one workgroup a CU.
        unsigned off = lane, off_last = in_last;
        int last = nblk - 1;
        asm volatile("" : "+v"(off), "+v"(off_last), "+s"(last));
        float best[kRows];
        int arg[kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r) { best[r] = DAGX_NEG_INF; arg[r] = lane; }
#pragma unroll
        for (int c0 = 0; c0 < kMaxBlocksFast; c0 += kCols) {
            if (c0 >= nblk) break;
            float x[kCols][kRows];   // all requested before any is looked at
#pragma unroll
            for (int c = 0; c < kCols; ++c)
#pragma unroll
                for (int r = 0; r < kRows; ++r) {
                    const int t = t0 + r < n_max ? t0 + r : n_max - 1, blk = min(c0 + c, last);
                    const float *from = A + (int64_t)(t + 1) * L + blk * kWave;
                    x[c][r] = from[blk < last ? off : off_last];
                }
#pragma unroll
            for (int c = 0; c < kCols; ++c)
#pragma unroll
                for (int r = 0; r < kRows; ++r) {
                    const int j = (c0 + c) * kWave + lane;
                    const float v = x[c][r] + to_end[c0 + c];   // (from node Lb on -inf or, where a cell was not written, NaN: never taken)
                    if (v > best[r]) { best[r] = v; arg[r] = j; }
                }
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            float top;
            const int j0 = wave_first_argmax(best[r], arg[r], top);
            if (lane == 0 && t0 + r < n_max) { sbest[t0 + r] = top; sidx[t0 + r] = j0; }
        }
    }
    __syncthreads();
    // best length: score / (t+1)^beta, first index among equals
    if (wave == 0) {
        float best = DAGX_NEG_INF;
        int arg = lane;
        for (int t = lane; t < n_max; t += kWave) {
            const float q = sbest[t] / a.penalty[t];
            if (q > best) { best = q; arg = t; }
        }
        float top;
        const int t_star = wave_first_argmax(best, arg, top);
        if (lane == 0) { a.pred_length[b] = t_star + 1; walk[t_star] = sidx[t_star]; s_star = t_star; }
    }
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(s_star) + 1;
    // table row s = t + 1 holds reach_t
    // (a path of finite score never meets a cell without a finite candidate)
    walk_back<TL, kDecodeThreads, true, STAGED>(A, srcblk, spitch, links, L, translen, n, __builtin_amdgcn_readfirstlane(sidx[n - 1]), 1,
                                        reinterpret_cast<WalkStage *>(lds_walk), [&](int s, int j) { walk[s - 1] = j; });
    if (wave != 0) return;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    // tokens: the last one always stays, an earlier one when it is not the pad and differs from its successor
    int count = 0;
    for (int k0 = 0; k0 < n_max; k0 += kWave) {
        const int k = k0 + lane;
        const bool in = k < n;
        const int node = in ? walk[k] : 0;
        const int64_t y = in ? tok[node] : a.pad;
        const int64_t ynext = (k + 1 < n) ? tok[walk[k + 1]] : a.pad;
        const bool keep = in && (k == n - 1 || (y != a.pad && y != ynext));
        const unsigned long long mask = __ballot(keep);
        const int pos = count + __popcll(mask & ((1ull << lane) - 1ull));
        if (keep) out_tokens[pos] = y;
        if (k < n_max) nodes[k] = in ? node : -1;
        count += __popcll(mask);
    }
    if (lane == 0) a.out_count[b] = count;
    for (int k = count + lane; k < n_max; k += kWave) out_tokens[k] = a.pad;
}

template <typename TL>
static int prepare_select() {
    static std::atomic<unsigned long long> done{0};
    return raise_lds_limit(reinterpret_cast<const void *>(viterbi_select_kernel<TL, true>), kWalkLds, done, "dag_viterbi_decode");
}

// What dagx_prepare_device does for the kernels of this file.
template <typename TL>
static int prepare_walks() {
    int rc = prepare_backtracks<float, TL>();
    if (!rc) rc = prepare_backtracks<__half, TL>();
    if (!rc) rc = prepare_backtracks<bf16_t, TL>();
    if (!rc) rc = prepare_align_chunks<float, TL, 1>();
    if (!rc) rc = prepare_align_chunks<float, TL, 2>();
    if (!rc) rc = prepare_align_chunks<__half, TL, 1>();
    if (!rc) rc = prepare_align_chunks<__half, TL, 2>();
    if (!rc) rc = prepare_align_chunks<bf16_t, TL, 1>();
    if (!rc) rc = prepare_align_chunks<bf16_t, TL, 2>();
    return rc ? rc : prepare_select<TL>();
}
int prepare_align_kernels() {
    int rc = prepare_walks<float>();
    if (!rc) rc = prepare_walks<__half>();
    return rc ? rc : prepare_walks<bf16_t>();
}

// workspace: [table B*T*L f32 | sync 16 + B*C | flags B | pad to 16 bytes | srcblk B*T*pitch bytes | match rows B*3*L f32]
static size_t decode_words(int B, int T, int L, int translen, int C) {
    return (size_t)B * T * L + 16 + (size_t)B * (C > 0 ? C : 1) + (size_t)B + 4 + (size_t)B * T * srcblk_pitch(L) / 4 + (size_t)B * 3 * L;
}
size_t decode_workspace_bytes(int B, int max_length, int L, int translen) {
    return decode_words(B, max_length + 1, L, translen, align_groups(B, max_length + 1, L, translen)) * 4;
}

template <typename TL>
static int launch_decode(const void *links, const float *node_logp, const int64_t *node_tokens, const int64_t *out_len,
                         int B, int L, int translen, int max_length, const float *penalty, int joint, int64_t pad,
                         int64_t *out_tokens, int64_t *out_count, int64_t *pred_length, int64_t *nodes,
                         void *workspace, hipStream_t st) {
    const int T = max_length + 1;
    int C = align_groups(B, T, L, translen);
    const int Cw = C > 0 ? C : 1;
    if (force_log_domain()) C = 0;
    float *table = static_cast<float *>(workspace);
    int *sync = reinterpret_cast<int *>(table + (size_t)B * T * L);
    int *flags = sync + 16 + B * Cw;
    unsigned char *srcblk = reinterpret_cast<unsigned char *>((reinterpret_cast<uintptr_t>(flags + B) + 15) & ~(uintptr_t)15);
    float *match3 = reinterpret_cast<float *>(srcblk + (size_t)B * T * srcblk_pitch(L));
    const int nsync = 16 + B * Cw;
    const int nprep = B * L > nsync ? B * L : nsync;
    hipLaunchKernelGGL(viterbi_prep_kernel, dim3((nprep + 255) / 256), dim3(256), 0, st, sync, nsync, flags, C > 0 ? 0 : 1,
                       node_logp, B, L, joint, match3);
    int rc = check_launch("viterbi_prep");
    if (rc) return rc;
    if (C > 0) {
        AlignTileArgs ta{};
        ta.match = match3; ta.ms0 = 3 * (int64_t)L; ta.ms1 = L; ta.ms2 = 1; ta.links = links;
        ta.out_len = out_len; ta.tgt_len = nullptr; ta.B = B; ta.T = T; ta.L = L; ta.translen = translen;
        ta.table = table; ta.sync = sync; ta.flags = flags; ta.srcblk = srcblk;
        ta.C = C; ta.mcap = 2; ta.decode = 1;
        if ((rc = launch_align_sweep<float, TL>(ta, "viterbi_sweep", st))) return rc;
    }
    constexpr int NT = 1024;
    hipLaunchKernelGGL((viterbi_table_kernel<TL, NT>), dim3(B), dim3(NT), (size_t)L * 8, st, match3, static_cast<const TL *>(links),
                       out_len, flags, T, L, translen, table, srcblk);
    if ((rc = check_launch("viterbi_table"))) return rc;
    DecodeArgs d{table, srcblk, links, out_len, node_tokens, penalty, T, L, translen, max_length, pad,
                 out_tokens, out_count, pred_length, nodes};
    const bool staged = staged_decode(B);
    auto select = staged ? viterbi_select_kernel<TL, true> : viterbi_select_kernel<TL, false>;
    if (staged && (rc = prepare_select<TL>())) return rc;
    hipLaunchKernelGGL(select, dim3(B), dim3(kDecodeThreads), staged ? kWalkLds : 0, st, d);
    return check_launch("viterbi_select");
}

}  // namespace dagx

using namespace dagx;

extern "C" int dagx_best_alignment(const void *match, int match_dtype, const int64_t match_strides[3],
                                   const void *links, int links_dtype,
                                   const int64_t *out_len, const int64_t *tgt_len,
                                   int B, int T, int L, int translen,
                                   int64_t *path, void *workspace, size_t workspace_bytes, void *stream) {
    if (B < 0 || T < 1 || L < 1 || translen < 1) { set_error("dag_best_alignment: bad sizes B=%d T=%d L=%d translen=%d", B, T, L, translen); return DAGX_ERR_ARGUMENT; }
    if (B == 0) return DAGX_OK;                 // an empty batch owns no memory: nothing to check or launch
    if (!match || !match_strides || !links || !out_len || !tgt_len || !path) { set_error("dag_best_alignment: null pointer argument"); return DAGX_ERR_ARGUMENT; }
    if (match_dtype < DAGX_F32 || match_dtype > DAGX_BF16 || links_dtype < DAGX_F32 || links_dtype > DAGX_BF16) { set_error("dag_best_alignment: unsupported dtype"); return DAGX_ERR_ARGUMENT; }
    if (L > 8192) { set_error("dag_best_alignment: graph size L=%d exceeds the supported 8192", L); return DAGX_ERR_UNSUPPORTED; }
    size_t need = align_workspace_bytes(B, T, L, translen);
    if (need > 0 && (!workspace || workspace_bytes < need)) { set_error("dag_best_alignment: workspace of %zu bytes required, %zu given", need, workspace_bytes); return DAGX_ERR_WORKSPACE; }
    AlignArgs a{match, match_strides[0], match_strides[1], match_strides[2], links, out_len, tgt_len,
                B, T, L, translen, path, nullptr};
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (match_dtype) {
        case DAGX_F32: return dispatch_align<float>(links_dtype, a, workspace, st);
        case DAGX_F16: return dispatch_align<__half>(links_dtype, a, workspace, st);
        default: return dispatch_align<bf16_t>(links_dtype, a, workspace, st);
    }
}

extern "C" int dagx_viterbi_decode(const void *links, int links_dtype, const float *node_logp, const int64_t *node_tokens,
                                   const int64_t *out_len, int B, int L, int translen, int max_length,
                                   const float *length_penalty, int joint, int64_t pad,
                                   int64_t *out_tokens, int64_t *out_count, int64_t *pred_length, int64_t *nodes,
                                   void *workspace, size_t workspace_bytes, void *stream) {
    if (B < 0 || L < 1 || translen < 1 || max_length < 1) { set_error("dag_viterbi_decode: bad sizes B=%d L=%d translen=%d max_length=%d", B, L, translen, max_length); return DAGX_ERR_ARGUMENT; }
    if (B == 0) return DAGX_OK;
    if (!links || !node_logp || !node_tokens || !out_len || !length_penalty || !out_tokens || !out_count || !pred_length || !nodes) { set_error("dag_viterbi_decode: null pointer argument"); return DAGX_ERR_ARGUMENT; }
    if (links_dtype < DAGX_F32 || links_dtype > DAGX_BF16) { set_error("dag_viterbi_decode: unsupported dtype"); return DAGX_ERR_ARGUMENT; }
    if (L > kMaxBlocksFast * kBlk) { set_error("dag_viterbi_decode: graph size L=%d exceeds the supported %d", L, kMaxBlocksFast * kBlk); return DAGX_ERR_UNSUPPORTED; }
    if (max_length + 1 > kDecodeMaxSteps) { set_error("dag_viterbi_decode: max_length=%d exceeds the supported %d", max_length, kDecodeMaxSteps - 1); return DAGX_ERR_UNSUPPORTED; }
    if ((int64_t)B * (max_length + 1) * L > 0x7fffffffLL) { set_error("dag_viterbi_decode: B*(max_length+1)*L too large for one call"); return DAGX_ERR_UNSUPPORTED; }
    const size_t need = decode_workspace_bytes(B, max_length, L, translen);
    if (!workspace || workspace_bytes < need) { set_error("dag_viterbi_decode: workspace of %zu bytes required, %zu given", need, workspace_bytes); return DAGX_ERR_WORKSPACE; }
    hipStream_t st = static_cast<hipStream_t>(stream);
#define DAGX_GO(TL) launch_decode<TL>(links, node_logp, node_tokens, out_len, B, L, translen, max_length, length_penalty, joint, pad, \
                                      out_tokens, out_count, pred_length, nodes, workspace, st)
    switch (links_dtype) {
        case DAGX_F32: return DAGX_GO(float);
        case DAGX_F16: return DAGX_GO(__half);
        default: return DAGX_GO(bf16_t);
    }
#undef DAGX_GO
}

extern "C" size_t dagx_workspace_bytes(int op, int B, int T, int L, int translen) {
    if (B <= 0 || T <= 0 || L <= 0) return 0;
    if (op == DAGX_OP_VITERBI_DECODE) return L <= kMaxBlocksFast * kBlk ? decode_workspace_bytes(B, T, L, translen) : 0;
    if (op == DAGX_OP_BEST_ALIGNMENT) return align_workspace_bytes(B, T, L, translen);
    if (op == DAGX_OP_BEST_ALIGNMENT_F64) return align_f64_workspace_bytes(B, T, L);
    if (op == DAGX_OP_LOSS_FWD) return loss_fwd_workspace_bytes(B, T, L, translen);
    if (op == DAGX_OP_LOSS_BWD) return loss_bwd_workspace_bytes(B);
    return 0;
}
