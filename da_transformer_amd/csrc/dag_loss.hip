// DAG loss on gfx950: log-semiring alpha/beta sweeps and the two gradient kernels.
//
//   alpha[t][j] = LSE_{i<j, j-i<=translen}(alpha[t-1][i] + E[i][j]) + match[t][j],  alpha[0][0] = match[0][0]
//   beta [t][i] = LSE_{j>i, j-i<=translen}(E[i][j] + beta[t+1][j]) + match[t][i],   beta[T_b-1][L_b-1] = match[..]
//   E[i][j] = links[i][j-i-1] ("shifted" layout), accumulation in fp32 whatever the input dtype.
//
// Both sweeps run in "position space": p = node for alpha, p = L_b-1-node for beta, step s = t for
// alpha, s = T_b-1-t for beta.  In that space both are the same recurrence over predecessors
// p' < p, start at p = 0 and are read out at (s, p) = (T_b-1, L_b-1).
//
// Storage of the sweep results (what the gradient kernels consume): positions are grouped in
// blocks of 64; every (step, block) has a float64 offset and every cell a float32 residual <= 0,
//   alpha[t][node] = off[t][p/64] + hat[t][node]          (hat indexed by node, off by position block)
// so the residuals keep full fp32 resolution no matter how negative the log-likelihood is.
//
// Two sweep implementations write this format:
//   * sweep_chunks_group ("fast"): exp(E) is staged once into registers as 64x64 tiles (lane <-> output position, 64
//     predecessors per tile).  Four steps at a time, what a block of positions receives from the blocks below it is a
//     product on the matrix cores; the 64x64 triangle on its diagonal is walked step by step by one wave.  The tiles of one
//     sweep are spread over a small pipeline of workgroups that hand the running vector on through global memory.
//     In float32 first; in float64 ("wide") for the samples whose float32 sweeps do not agree.
//   * dag_sweep_exact_kernel: every term evaluated in the log domain, one workgroup per sweep.
//     Handles any size and any dynamic range; it re-does the samples the others leave.
#include <atomic>
#include <cstdint>
#include <type_traits>

#include "dag_chunks.h"

namespace dagx {


struct SweepArgs {
    const void *match; int64_t ms0, ms1, ms2;
    const void *links;
    const int64_t *out_len, *tgt_len;
    int B, T, L, translen, NBK;
    float *hat[2];     // residual tables of the two sweeps of a sample (with gradients: alpha-hat, beta-hat)  [B][T][L]
    double *off[2];    // block offsets        [B][T][NBK]
    double *logz;      // [2][B] read-outs of the two sweeps (with gradients: alpha end, beta end)
    float *loss;       // [B] the read-out of sweep `loss_dir` in float
    int loss_dir;      // 0: first sweep's read-out (alpha), 1: second sweep's (beta: the partition function the backward divides by)
    int *flags;        // [B] 1 = sample must be (re)done (by the wide tile sweeps, then by the exact kernel); 2 = the wide sweeps settled it
    // fast path, all zero on entry and left zero: [0] ticket counter, [1] workgroups that have left, [2] samples the
    // float32 launch flagged (cleared by the wide launch),
    // [16 + (dir*B + b)*C + group] progress words, then [B] workgroups of the sample that have left, then [B] "risk"
    // words (a group of the sample gave up waiting for its producer)
    int *sync;
    int C;             // workgroups per sweep (fast path): the most of any table
    TableChoice choice; // (here, not behind the tables: what a kernel reads first lies in as few lines of the argument block as possible)
    int ndir;          // sweeps per sample in the tile kernel: always two, which bracket the result (see sweep_chunks_group)
    // The two tile sweeps of a sample: direction (0: alpha, 1: beta) and rounding side (0: every number too small
    // for the linear domain becomes 0, a lower bound of the sum over paths; 1: it becomes the smallest number the
    // domain holds, an upper bound).  With gradients {alpha/upper, beta/lower}, without {alpha/lower, alpha/upper}.
    unsigned char rev[2], upper[2];
    int only_flagged;  // exact kernel: 0 = every sample; 1 = samples whose flag is set
    double *zfast;     // [2][B] the fast kernel's own read-outs (never rewritten by the exact kernel)
};

struct TileSweepArgs : SweepArgs {
    GroupTable table[kMostTables];   // fast path, host-built
};

__device__ __forceinline__ bool lengths_ok(int Lb, int Tb, int L, int T) {
    return Tb >= 1 && Lb >= 1 && Tb <= T && Lb <= L && Tb <= Lb;
}

// A chunk of R terms held in registers, merged into (m,s): max pass, then exp-sum pass.  The terms and the
// running maximum are float64 (absolute log values of any magnitude),
// the exponentials of the differences and their sum float32.
template <int R>
__device__ __forceinline__ void lse_chunk_d(const double (&x)[R], double &m, float &s) {
    double cm = x[0];
#pragma unroll
    for (int r = 1; r < R; ++r) cm = fmax(cm, x[r]);
    if (cm == (double)DAGX_NEG_INF) {   // nothing finite here (fmax skips a NaN, which must not get lost)
        bool nan = false;
#pragma unroll
        for (int r = 0; r < R; ++r) nan |= x[r] != x[r];
        if (nan) s = __builtin_nanf("");
        return;
    }
    const double nm = fmax(m, cm);
    float part = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) part += fast_exp2((float)(x[r] - nm) * kLog2e);
    s = s * fast_exp2((float)(m - nm) * kLog2e) + part;  // m = -inf gives 0 * 0
    m = nm;
}

__device__ __forceinline__ double wave_max_d(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}

// ================================================================================================
// Exact sweep
// ================================================================================================

// One row of the table from this step's values by node (absolute, float64): per block of 64 positions the
// offset is the block maximum and the residuals are what is left, so that no cell's precision depends on
// how far it lies under the largest value of the row.
template <int NT>
__device__ __forceinline__ void write_row(const double *f, int dir, int Lb, int NBb, float *hat_row, double *off_row) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    for (int blk = wave; blk < NBb; blk += NT / kWave) {
        const int p = blk * kBlk + lane;
        const int node = dir ? Lb - 1 - p : p;
        const double v = p < Lb ? f[node] : (double)DAGX_NEG_INF;
        const double bm = wave_max_d(v);
        if (lane == 0) off_row[blk] = bm;
        if (p < Lb) hat_row[node] = bm > (double)DAGX_NEG_INF ? (float)(v - bm) : DAGX_NEG_INF;
    }
}

// Log-domain sweeps, one workgroup per (sample, direction).  The running vector is kept in float64 (LDS), every
// term is formed as a float64 sum and only the difference to the cell's own running maximum is exponentiated
// in float32: cells hundreds or thousands of nats under the largest value of their step, which is where the
// posterior mass of sharply peaked inputs can sit, keep the full precision of their inputs.
template <typename TM, typename TL, int NT>
__device__ __forceinline__ void exact_sweep_sample(const SweepArgs &a, const int b, const int dir, double *lds_x) {
    // lds_x: two vectors of L doubles;  dir 0: alpha, 1: beta
    const int tid = threadIdx.x;
    const int L = a.L, T = a.T, translen = a.translen;
    const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
    const TM *match = static_cast<const TM *>(a.match) + (int64_t)b * a.ms0;
    const TL *links = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    float *hat = a.hat[dir] + (int64_t)b * T * L;
    double *off = a.off[dir] + (int64_t)b * T * a.NBK;
    double *fprev = lds_x, *fcur = lds_x + L;

    if (!lengths_ok(Lb, Tb, L, T)) {
        if (tid == 0) { a.logz[dir * a.B + b] = (double)DAGX_NEG_INF; if (dir == a.loss_dir) a.loss[b] = DAGX_NEG_INF; }
        return;
    }
    const int slack = Lb - Tb;  // band: s <= p <= slack + s
    const int NBb = (Lb + kBlk - 1) / kBlk;
    const int t0 = dir ? Tb - 1 : 0, start = dir ? Lb - 1 : 0;
    const float m0 = to_float(match[(int64_t)t0 * a.ms1 + (int64_t)start * a.ms2]);
    for (int j = tid; j < L; j += NT) fprev[j] = j == start ? (double)m0 : (double)DAGX_NEG_INF;
    __syncthreads();
    write_row<NT>(fprev, dir, Lb, NBb, hat + (int64_t)t0 * L, off + (int64_t)t0 * a.NBK);

    // A team of kTeam lanes works on one node; each of its lanes has R terms in flight.
    constexpr int kTeam = 8, R = 8;
    const int team = tid / kTeam, sub = tid % kTeam;
    auto team_merge = [](double &m, float &sum) {   // the lanes' (maximum, sum) pairs into one, in every lane of the team
#pragma unroll
        for (int o = kTeam / 2; o > 0; o >>= 1) {
            const double mo = __shfl_xor(m, o, kWave);
            const float so = __shfl_xor(sum, o, kWave);
            const double nm = fmax(m, mo);
            if (nm > (double)DAGX_NEG_INF)
                sum = sum * fast_exp2((float)(m - nm) * kLog2e) + so * fast_exp2((float)(mo - nm) * kLog2e);
            else
                sum += so;   // 0 + 0, or a NaN on its way
            m = nm;
        }
    };
    for (int s = 1; s < Tb; ++s) {
        const int t = dir ? Tb - 1 - s : s;
        if (dir == 0) {
            // A team of kTeam lanes <-> node j of the band; the team's lanes deal the predecessors i among
            // themselves (lane q takes i = ilo + q, ilo + q + kTeam, ...), R of them in flight per lane, and
            // merge their (maximum, sum) pairs by shuffles.  Teams of one wave hold neighbouring nodes, so a
            // wave-wide load reads kTeam runs of neighbouring elements; nodes are dealt to the teams round
            // robin, which mixes nodes with few and with many predecessors in every team.
            const int jhi = slack + s;
            for (int j = tid; j < L; j += NT)
                if (j < s || j > jhi) fcur[j] = (double)DAGX_NEG_INF;
            const unsigned rs = (unsigned)(translen - 1);   // E[i][j-i-1] sits at links[i*(translen-1) + j-1]: 32-bit offsets
            for (int j = s + team; j <= jhi; j += NT / kTeam) {
                const float mj = to_float(match[(int64_t)t * a.ms1 + (int64_t)j * a.ms2]);
                int ilo = j - translen; if (ilo < s - 1) ilo = s - 1;
                double m = (double)DAGX_NEG_INF; float sum = 0.f;
                const unsigned o_last = (unsigned)(j - 1) * (unsigned)translen;   // the offset of i = j-1, the largest
                unsigned o = (unsigned)(ilo + sub) * rs + (unsigned)(j - 1);
                for (int i0 = ilo + sub; i0 < j; i0 += kTeam * R, o += kTeam * R * rs) {
                    float e[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const unsigned oc = o + (unsigned)(r * kTeam) * rs;
                        e[r] = to_float(links[oc < o_last ? oc : o_last]);
                    }
                    double x[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {   // a term beyond the last predecessor: -inf through its transition
                        const int i = i0 + r * kTeam;
                        x[r] = fprev[i < j ? i : j - 1] + (double)(i < j ? e[r] : DAGX_NEG_INF);
                    }
                    lse_chunk_d<R>(x, m, sum);
                }
                team_merge(m, sum);
                if (sub == 0)
                    fcur[j] = (m > (double)DAGX_NEG_INF || sum != sum) ? (m + (double)(fast_log2(sum) * kLn2)) + (double)mj : (double)DAGX_NEG_INF;
            }
        } else {
            // the same with a team <-> node i and the team's lanes dealing the successors j among themselves: a
            // team reads runs of kTeam neighbouring elements of its node's row of links
            const int ilo_band = Lb - 1 - (slack + s), ihi_band = Lb - 1 - s;  // nodes whose position is in the band
            const int jtop = Lb - 1 - (s - 1), jbot = Lb - 1 - (slack + s - 1);  // band of the previous step
            for (int i = tid; i < L; i += NT)
                if (i < ilo_band || i > ihi_band) fcur[i] = (double)DAGX_NEG_INF;
            for (int i = ilo_band + team; i <= ihi_band; i += NT / kTeam) {
                const float mi = to_float(match[(int64_t)t * a.ms1 + (int64_t)i * a.ms2]);
                const int jmax = i + translen < jtop ? i + translen : jtop;
                const int jmin = i + 1 > jbot ? i + 1 : jbot;
                const unsigned rbase = (unsigned)i * (unsigned)translen - (unsigned)i - 1u;   // E[i][j-i-1] = links[rbase + j], modulo 2^32
                double m = (double)DAGX_NEG_INF; float sum = 0.f;
                for (int j0 = jmin + sub; j0 <= jmax; j0 += kTeam * R) {
                    float e[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int j = j0 + r * kTeam;
                        e[r] = to_float(links[rbase + (unsigned)(j <= jmax ? j : jmax)]);
                    }
                    double x[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int j = j0 + r * kTeam;
                        x[r] = fprev[j <= jmax ? j : jmax] + (double)(j <= jmax ? e[r] : DAGX_NEG_INF);
                    }
                    lse_chunk_d<R>(x, m, sum);
                }
                team_merge(m, sum);
                if (sub == 0)
                    fcur[i] = (m > (double)DAGX_NEG_INF || sum != sum) ? (m + (double)(fast_log2(sum) * kLn2)) + (double)mi : (double)DAGX_NEG_INF;
            }
        }
        __syncthreads();
        write_row<NT>(fcur, dir, Lb, NBb, hat + (int64_t)t * L, off + (int64_t)t * a.NBK);
        double *sw = fprev; fprev = fcur; fcur = sw;
    }
    if (tid == 0) {
        const double z = fprev[dir ? 0 : Lb - 1];
        a.logz[dir * a.B + b] = z;
        if (dir == a.loss_dir) a.loss[b] = (float)z;
    }
}

template <typename TM, typename TL, int NT>
__global__ __launch_bounds__(NT) void dag_sweep_exact_kernel(SweepArgs a) {
    extern __shared__ double lds_x[];
    if (a.only_flagged && a.flags[blockIdx.x] != 1) return;
    exact_sweep_sample<TM, TL, NT>(a, (int)blockIdx.x, (int)blockIdx.y, lds_x);
}

// ================================================================================================
// Tile sweeps: register-resident exp(E) tiles, pipelined workgroups
// ================================================================================================

// ---- the sweeps in chunks of four steps (geometry, tiles and products: dag_chunks.h) ---------------------------------
// What a step-by-step sweep pays per step -- barriers, LDS round trips, scales, a few hundred instructions a wave around
// the FMAs, 2.0 us at L = 512 -- is paid here once per four steps, and the tiles below the diagonal run on the matrix cores
// (float32: at twice the rate of DPP FMAs; float64: at their rate, but a transition is converted once per four steps).
// What is left on the critical path is the walk of one block through four steps (48 FMAs and 20 to 40 other instructions
// a step, 5.5 cycles each), the product of the tile next to the diagonal in front of it, and one stage per block of the
// graph.  (With that product a stage ahead, too, the stages are 600 cycles shorter but two per block: forward at B = 64,
// L = 512, T = 64 115 us instead of 107, L = 256 70 instead of 66, L = 128 52 instead of 56.)
//   step by step -> chunks, forward: B = 64, L = 512, T = 64 134 -> 106 us; L = 64 (T = 64) 81 -> 47; L = 256 99 -> 65;
//   B = 16, L = 1024, T = 256 572 -> 341; B = 64, L = 512, transitions of at most 32: 136 -> 77.
//   In float64: B = 16, L = 1024, T = 256 833 -> 512 us; B = 64, L = 512, T = 64 216 -> 150.
// What bounds it: a SIMD gives its cycles either to matrix instructions or to vector instructions, never to both
// (measured: a wave of DPP FMAs beside one of v_mfma_f32_4x4x1 advances only when that has ended, whatever their
// priorities), so that products, walks and the rest of a stage add up.
// A walking wave loads and converts its own match rows and writes its own results (as duties of other waves, through
// LDS, they cost those waves more than they save it).
//
// Inter-workgroup hand-over of the running vector (the groups of one sweep form a one-way pipeline): a producer writes its
// table rows (hat, off) with agent-scope stores and raises its progress word when the waves of its last two blocks have
// both seen theirs of the last stage complete, early in the next one; a consumer copies the rows of a chunk (global ->
// LDS) when the word covers it: of the block right below it one stage before its first block walks that chunk, of the
// others two.  (All of them two stages ahead, and the word raised half a stage later: four stages a hand-over instead of
// one and a half, B = 16, L = 1024, T = 64 189 us instead of 159.)  Every wait is bounded: on expiry the sample is
// marked for the log-domain kernel and the group leaves.
//
// Leaving: every workgroup counts itself out of its sample and out of the launch.  The last one of a sample compares the
// two read-outs, sets the sample's flag (1 = still to be done) and clears the sample's pipeline words; the last one of
// the launch clears the ticket counter -- so the words are all zero again when the launch is over and need no fill in
// front of it.
template <typename TM, typename TL, bool WIDE>
__device__ __forceinline__ void sweep_chunks_group(const TileSweepArgs &a, const GroupTable &plan, const int b, const int slot, const int g,
                                                   float *lds_raw, int *gstart, int *s_abort_p) {
    using CH = Chunks<WIDE>;
    using Cell = typename CH::Cell;
    // slot: which of the sample's two sweeps (its tables, pipeline words and read-out); dir: its direction;
    // upper: its rounding side.  The linear domain flushes what is too far under its scale -- a transition, a cell under
    // its block maximum, a block under the largest of its neighbours, a product of such numbers.  The lower sweep lets all
    // of that become 0, so its read-out never exceeds log Z; the upper sweep puts the smallest normal number (or a constant
    // that covers every flushed product) in its place, so its read-out never falls short of log Z.  The sample's result
    // stands when the two read-outs agree; what was flushed then carried no mass that matters, wherever it was flushed.
    const int dir = a.rev[slot];
    const bool upper = a.upper[slot] != 0;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int C = a.C;
    int *risk = a.sync + 16 + a.ndir * a.B * C + a.B + b;
    // (through opaque_uniform: else the compiler reads them from the argument block again in every stage, a scalar-memory
    //  round trip each)
    const int L = opaque_uniform(a.L), T = a.T, translen = a.translen, NBK = opaque_uniform(a.NBK);
    const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
    if (!lengths_ok(Lb, Tb, L, T)) {
        if (g == 0 && tid == 0) { a.logz[slot * a.B + b] = (double)DAGX_NEG_INF; if (slot == a.loss_dir) a.loss[b] = DAGX_NEG_INF; store_agent(a.zfast + slot * a.B + b, (double)DAGX_NEG_INF); }
        return;
    }
    const TM *match = static_cast<const TM *>(a.match) + (int64_t)b * a.ms0;
    const TL *links = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    float *hat = a.hat[slot] + (int64_t)b * T * L;
    double *off = a.off[slot] + (int64_t)b * T * NBK;
    int *prog = a.sync + 16 + (slot * a.B + b) * C;

    const int t_first = dir ? Tb - 1 : 0, node_first = dir ? Lb - 1 : 0;
    const float m0 = to_float(match[(int64_t)t_first * a.ms1 + (int64_t)node_first * a.ms2]);
    const int slack = Lb - Tb;                    // band: s <= p <= slack + s
    const int NBb = (Lb + kBlk - 1) / kBlk;
    const int W = (translen + kBlk - 1) / kBlk;
    if (tid <= C) gstart[tid] = plan.gtab[NBb][tid];
    __syncthreads();
    const int jb0 = __builtin_amdgcn_readfirstlane(gstart[g]), jb1 = __builtin_amdgcn_readfirstlane(gstart[g + 1]);
    int last_group = 0;
    for (int q = 0; q < C; ++q) if (gstart[q + 1] > gstart[q]) last_group = q;
    last_group = __builtin_amdgcn_readfirstlane(last_group);
    if (jb0 >= jb1) return;                       // nothing to do for this group (short sample); nobody waits on it
    const int nblk = jb1 - jb0;
    const int flo = tile_ilo(jb0, W);             // lowest foreign block this group ever reads
    const bool producer = g < last_group, consumer = flo < jb0;
    const ChunkLds o = chunk_lds(jb0, nblk, W, WIDE);
    int ntile = 0;
    for (int q = 0; q < nblk; ++q) ntile += tiles_of_block<1>(jb0 + q, W);
    if (nblk > kChunkBlocks || ntile > kTileCap - nblk || o.total * 4 > kChunkLdsBytes) {   // cannot happen with the host's partition
        if (tid == 0) { store_agent(risk, 1); store_agent(prog + g, 1 << 30); }
        return;
    }
    const bool owner = wave < nblk;               // this wave walks block jb0 + wave
    const int helpers = kTileWaves - nblk;

    const TileDeal deal = plan.deal[NBb][g];
    const WaveTiles t = plan_wave<1>(deal, jb0, nblk, W, o.runs, wave, lane);
    // A consumer group has nothing to do for the first stages: it lets the first group of its sweep have the memory's
    // bandwidth for its tiles.  (Progress words: 1 once the group's tiles are staged, then 2 + n when the rows of the first n
    // chunks of its last block and n + 1 of the others are in memory -- and so, since it has read them, n of all blocks below.)
    if (consumer) {
        if (wave == 0)
            for (int spins = 0; spins < kSpinLimit && __builtin_amdgcn_readfirstlane(load_agent(prog)) < 1; ++spins) __builtin_amdgcn_s_sleep(8);
        __syncthreads();
    }
    const unsigned lds_base = (unsigned)reinterpret_cast<uintptr_t>(lds_raw);
    float *const patch = lds_raw + wave * (kBlk * kPatchPitch);
    const int last_index = L * translen - 1;
    const float tiny = !upper ? 0.f : kTinyStored;
    auto elements = [&](const int samples) { const int64_t n = (int64_t)samples * L * translen; return n < (1 << 28) ? (int)n : 1 << 28; };
    const int before = elements(b), behind = elements(a.B - 1 - b);
    auto stage = [&](const int u) __attribute__((always_inline)) {
        stage_tile<TL, CH::kLinkShift, true, 8>(patch, links, t.I[u], jb0 + t.q[u], lane, dir, Lb, translen, last_index, before, behind, tiny);
    };
    Tile t0, t1, t2;
    auto read = [&](Tile &tile, const bool triangle) __attribute__((always_inline)) {
        if (!WIDE || triangle) read_patch(tile, patch, lane, dir); else read_patch_wide(tile, patch, lane, dir);
    };
    if (t.ok[0] || t.adjacent) { stage(0); read(t0, false); }
    if (t.ok[1]) { stage(1); read(t1, false); }
    if (t.ok[2] || owner) { stage(2); read(t2, owner); }
    if (owner) fold_triangle(t2, lane);
    __syncthreads();   // every wave is done with its transpose patch: the LDS now holds the buffers of the stages
    if (producer && g == 0 && tid == 0) store_agent(prog, 1);

    int *const lds_i = reinterpret_cast<int *>(lds_raw);
    int *const published_by = lds_i + o.both;
    if (tid == 0) *published_by = 0;
    const int D = o.depth;
    // ---- step 0: only position 0 is alive ----
    // exp(m): fraction in [1, 2) and exponent; what no such pair holds as in the constants above, +inf and NaN as NaN
    auto split_exp = [&](const float m, float &frac, int &exp) __attribute__((always_inline)) {
        const float hi = m * kLog2e;
        const float fl = __builtin_floorf(hi);
        // (the product's rounding error and log2(e)'s own: for a match of -60 they are worth 3e-6 of the cell)
        const float lo = __builtin_fmaf(m, kLog2e, -hi) + m * 1.925963033500e-08f;
        float f = fast_exp2((hi - fl) + lo);
        int n = (int)__builtin_amdgcn_fmed3f(fl, -(float)kMatchExpMax, (float)kMatchExpMax);
        if (!(hi >= -(float)kMatchExpMax)) f = upper ? 1.f : 0.f;
        if (m == DAGX_NEG_INF) f = 0.f;
        if (!(hi <= (float)kMatchExpMax)) { f = __builtin_nanf(""); n = 0; }
        frac = f; exp = n;
    };
    float f0; int n0;
    split_exp(m0, f0, n0);
    n0 = __builtin_amdgcn_readfirstlane(n0);
    const bool alive0 = !(f0 == 0.f);     // (a NaN is on its way)
    Cell *const eb = reinterpret_cast<Cell *>(lds_raw + o.eb), *const part = reinterpret_cast<Cell *>(lds_raw + o.part);
    auto pow2 = [](const Cell x, const int n) __attribute__((always_inline)) { if constexpr (WIDE) return __builtin_ldexp(x, n); else return __builtin_ldexpf(x, n); };
    for (int q = wave; q < nblk; q += kTileWaves) {
        const int Jb = jb0 + q, p = Jb * kBlk + lane;
        const bool here = p == 0 && alive0;
        eb[(jb0 - flo + q) * D * 256 + cell_place<WIDE>(lane)] = here ? pow2((Cell)f0, CH::kShift - 1) : (Cell)0;
        if (lane == 0) lds_i[o.kap + (jb0 - flo + q) * D * 4] = here ? n0 + 1 : kDeadExp;
        if (p < Lb) store_agent(hat + (int64_t)t_first * L + (dir ? Lb - 1 - p : p), here ? (fast_log2(f0) - 1.f) * kLn2 : DAGX_NEG_INF);
        if (lane == 0) store_agent(off + (int64_t)t_first * NBK + Jb, Jb == 0 && alive0 ? (double)(n0 + 1) * 0.6931471805599453 : (double)DAGX_NEG_INF);
    }
    if (tid < 2 * 256) part[o.runs * 2 * 256 + tid] = (Cell)0;
    if (tid < nblk * 2 * kChunk) lds_i[o.part_scale + tid] = kDeadExp;   // (stays with a block without such tiles)
    if (Tb == 1 && tid == 0 && jb0 == 0) {
        const double z = (Lb == 1 && alive0) ? (double)m0 : (double)DAGX_NEG_INF;
        a.logz[slot * a.B + b] = z; if (slot == a.loss_dir) a.loss[b] = (float)z; store_agent(a.zfast + slot * a.B + b, z);
    }
    const char *hat_c = reinterpret_cast<const char *>(hat);
    const char *off_c = reinterpret_cast<const char *>(off);
    const char *match_c = reinterpret_cast<const char *>(match);
    const unsigned long long hat_u = uniform_address(hat), off_u = uniform_address(off);
    const int ms1 = opaque_uniform((int)a.ms1), ms2 = opaque_uniform((int)a.ms2);   // the host checked that match indices fit 32 bits
    const int NC = (Tb - 1 + kChunk - 1) / kChunk;  // chunks of steps 1 .. T_b-1
    const int floor_exp = upper ? CH::kFloor : CH::kFloor - 1;   // see pow2_clamped
    const Cell tiny_up = upper ? (WIDE ? (Cell)2.2250738585072014e-308 : (Cell)kTinyStored) : (Cell)0;   // 2^kFloor
    // more than everything that may have been flushed on the way to a block's sum: 64 products a tile under 2^kFloor
    // each, 16 tiles, as many scaled sums
    const Cell flush_up = upper ? (WIDE ? (Cell)9.332636185032189e-302 : (Cell)2.4074124e-35f) : (Cell)0;
    auto opaque_lane = [&] { int x = tid & (kWave - 1); asm volatile("" : "+v"(x)); return x; };
    // a block's chunks with a live cell (4c+1 .. 4c+4 meets the block's band), and its chunks as a source (4c .. 4c+3)
    auto dest_lo = [&](const int J) { return 16 * J - 1 - (slack >> 2); };
    auto dest_hi = [&](const int J) { return 16 * J + 15; };
    auto src_lo = [&](const int I) { return 16 * I - ((slack + 3) >> 2); };

    // ---- the foreign blocks whose table rows this wave fetches ----
    int f_blk[kForeign], f_first, f_count;
    wave_foreign(deal, wave, f_first, f_count);
#pragma unroll
    for (int u = 0; u < kForeign; ++u) f_blk[u] = u < f_count ? flo + f_first + u : -1;
    // Table rows of steps 4c .. 4c+3 of a foreign block (complete: 64 positions): one copy of sixteen bytes a lane for the
    // residuals (row lane / 16, in the order of the nodes), one for the offsets.
    auto request_rows = [&](const int I, const int c, const int lane) __attribute__((always_inline)) {
        auto row_of = [&](const int k) { const int s = kChunk * c + k, sc = s < Tb ? s : Tb - 1; return dir ? Tb - 1 - sc : sc; };
        const int node = (dir ? Lb - kBlk - I * kBlk : I * kBlk) + 4 * (lane & 15);
        dma_dwordx4_agent_u(lds_base + (unsigned)(o.frows + (I - flo) * 256) * 4u, hat_u, (unsigned)(row_of(lane >> 4) * L + node) * 4u);
        dma_dword_agent_u(lds_base + (unsigned)(o.foff + (I - flo) * 64) * 4u, off_u,
                          (unsigned)(row_of((lane >> 1) & 3) * NBK + I) * 8u + (unsigned)(lane & 1) * 4u);
    };
    // ... as cells, four positions of one step a lane
    auto convert_rows = [&](const int I, const int sl, const int lane) __attribute__((always_inline)) {
        const int at = I - flo;
        const float *const row = lds_raw + o.frows + at * 256 + (lane & 3) * kBlk;
        const double v = reinterpret_cast<const double *>(lds_raw + o.foff + at * 64)[lane & (kChunk - 1)];
        if constexpr (WIDE) {
            // positions 8 (lane / 16) + (lane / 4 mod 4) + {0, 4, 32, 36}: two neighbours of a product's first operand each
            typedef double f64x2 __attribute__((ext_vector_type(2)));
            const int r = 8 * (lane >> 4) + ((lane >> 2) & 3);
            const float *const src = row + (dir ? kBlk - 1 - r : r);
            f64x2 *const dst = reinterpret_cast<f64x2 *>(eb + (at * D + sl) * 256) + lane;
            const int pitch = dir ? -4 : 4;
            double w[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float x = src[pitch * (q < 2 ? q : q + 6)];
                const float hi = x * kLog2e, n = __builtin_floorf(hi), lo = __builtin_fmaf(x, kLog2e, -hi) + x * 1.925963033500e-08f;
                const double z = __builtin_ldexp((double)fast_exp2((hi - n) + lo), (int)__builtin_fmaxf(n, -4000.f) + CH::kShift);
                w[q] = x == DAGX_NEG_INF ? 0.0 : z + tiny_up;
            }
            dst[0] = f64x2{w[0], w[1]};
            dst[64] = f64x2{w[2], w[3]};
        } else {
            // lane 4 (i & 15) + step has the positions 16 q + (i & 15)
            const float *const src = row + (dir ? kBlk - 1 - (lane >> 2) : lane >> 2);
            const int pitch = dir ? -16 : 16;
            float x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = src[q * pitch];
            f32x4 ev;
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] *= kLog2e;
            if (__builtin_amdgcn_ballot_w64(!(fminf(fminf(x[0], x[1]), fminf(x[2], x[3])) >= -115.f)) == 0) {   // (as exp2_shifted above -115)
#pragma unroll
                for (int q = 0; q < 4; ++q) ev[q] = __builtin_ldexpf(fast_exp2(x[q]), kShift2);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float w = exp2_shifted(x[q]);
                    ev[q] = (x[q] > -3.0e38f && w < (float)tiny_up) ? (float)tiny_up : w;
                }
            }
            *reinterpret_cast<f32x4 *>(eb + (at * D + sl) * 256 + lane * 4) = ev;
        }
        const int kp = v > (double)DAGX_NEG_INF ? (int)__builtin_rint(v * 1.4426950408889634) : kDeadExp;
        if (lane < kChunk) lds_i[o.kap + (at * D + sl) * 4 + lane] = kp;
    };

    // ---- the stages ----
    const int first_stage = consumer ? -2 : -1, end_stage = NC - 1 + nblk - 1;
    const int *below = prog + (g > 0 ? g - 1 : 0);
    // stages in which a tile's block takes part, and those in which the tile's source has a live cell
    int t_from[kTilesPerWave], t_to[kTilesPerWave], t_src_from[kTilesPerWave], t_src_to[kTilesPerWave];
    int t_shift[kTilesPerWave], t_cells[kTilesPerWave], t_kaps[kTilesPerWave], t_scale_at[kTilesPerWave], t_scales[kTilesPerWave];
#pragma unroll
    for (int u = 0; u < kTilesPerWave; ++u) {
        const int J = jb0 + t.q[u], at = t.q[u] - 1, lo = tile_ilo(J, W);   // chunk = stage - at
        t_from[u] = at + (dest_lo(J) > 0 ? dest_lo(J) : 0);
        t_to[u] = t.ok[u] ? at + (dest_hi(J) < NC - 1 ? dest_hi(J) : NC - 1) : -100;
        t_src_from[u] = at + src_lo(t.I[u]); t_src_to[u] = at + dest_hi(t.I[u]);
        t_shift[u] = (((-at) % D) + D) % D;
        t_cells[u] = (t.I[u] - flo) * D * 256; t_kaps[u] = o.kap + (t.I[u] - flo) * D * 4;
        t_scale_at[u] = o.kap + (lo - flo) * D * 4; t_scales[u] = J - 1 - lo;
    }
    if (NC == 0) return;
    __syncthreads();

    // One barrier a stage; a loop for each kind of wave, so that the registers hold what that kind needs.
    auto stages = [&](auto walks, auto fetches) __attribute__((always_inline)) {
        constexpr bool WALKS = decltype(walks)::value, FETCHES = decltype(fetches)::value;
        // ring slots: chunk c of a block's cells is in slot c mod D (ring: the stage mod D)
        int slot_own = 0, seen = 0, requested = first_stage - 1, ring = ((first_stage % D) + D) % D;
        auto next_slot = [&](const int x) { return x + 1 == D ? 0 : x + 1; };
        // the walking wave's state: the last step's cells and their exponent; the next chunk's match rows as loaded, then
        // exp(match) relative to the rows' exponents N
        const int J = jb0 + wave, first = J * kBlk, own_src = jb0 - flo + wave;
        // (float64: a fraction and its exponent relative to N)
        Cell e = 0;
        int kap = kDeadExp, N[kChunk] = {0, 0, 0, 0}, mt_exp[kChunk] = {0, 0, 0, 0};
        float mt[kChunk] = {0.f, 0.f, 0.f, 0.f};
        TM raw[kChunk];
        if (WALKS && J == 0) {
            if (lane == 0 && alive0) e = pow2((Cell)f0, CH::kShift - 1);
            kap = alive0 ? n0 + 1 : kDeadExp;
        }
        auto load_match = [&](const int c, const int lane) __attribute__((always_inline)) {
            const int p = first + lane, pc = p < Lb ? p : Lb - 1, s0 = kChunk * c + 1;
            const unsigned lane_off = (unsigned)((dir ? Lb - 1 - pc : pc) * ms2) * (unsigned)sizeof(TM);
            const char *row = match_c + (unsigned)((dir ? Tb - 1 - s0 : s0) * ms1) * (unsigned)sizeof(TM);
            const int step = (dir ? -ms1 : ms1) * (int)sizeof(TM);
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                raw[k] = *reinterpret_cast<const TM *>(row + lane_off);
                if (s0 + k + 1 < Tb) row += step;      // (rows past the last step: the last one again)
            }
        };
        // (with_pair: the walked chunk's fold_two is reduced along with the match rows)
        auto convert_match = [&](const int c, const int lane, auto with_pair, float &pair) __attribute__((always_inline)) {
            const int s0 = kChunk * c + 1;
            float m[kChunk], top[kChunk];
#pragma unroll
            for (int k = 0; k < kChunk; ++k) m[k] = to_float(raw[k]);
            // in the band: s <= p <= slack + s (mostly the whole block, in all four steps)
            if (!(first >= s0 + kChunk - 1 && first + kBlk - 1 <= slack + s0 && s0 + kChunk <= Tb)) {
                const int d0 = first + lane - s0;
#pragma unroll
                for (int k = 0; k < kChunk; ++k)
                    m[k] = (unsigned)(d0 - k) < (s0 + k < Tb ? (unsigned)slack + 1u : 0u) ? m[k] : DAGX_NEG_INF;
            }
#pragma unroll
            for (int k = 0; k < kChunk; ++k) top[k] = m[k];
            wave64_max4<decltype(with_pair)::value>(top, pair);
            float log2e = kLog2e;
            asm("" : "+v"(log2e));                    // (an instruction takes one scalar register: N)
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                // relative to the row's exponent: its largest cell becomes a number in (1/2, 1]
                const float n = __builtin_amdgcn_fmed3f(__builtin_ceilf(top[k] * kLog2e), -(float)kMatchExpMax, (float)kMatchExpMax);
                N[k] = __builtin_amdgcn_readlane((int)n, 63);
                if constexpr (WIDE) {
                    split_exp(m[k], mt[k], mt_exp[k]);
                    mt_exp[k] -= N[k];
                } else mt[k] = __builtin_fmaf(m[k], log2e, -lane_bcast(n, 63));
            }
            if constexpr (WIDE) return;
            if (__builtin_amdgcn_ballot_w64(!(fminf(fminf(mt[0], mt[1]), fminf(mt[2], mt[3])) >= -126.f)) != 0 && upper) {
#pragma unroll
                for (int k = 0; k < kChunk; ++k) mt[k] = m[k] > DAGX_NEG_INF && mt[k] < -126.f ? -126.f : mt[k];
            }
#pragma unroll
            for (int k = 0; k < kChunk; ++k) mt[k] = fast_exp2(mt[k]);
        };
        // the chunk just walked (cells v, exponents kk; kept: the largest of its steps 0 and 2) into the tables
        auto write_out = [&](const int c, const Cell (&v)[kChunk], const int (&kk)[kChunk], const float kept, const int lane) __attribute__((always_inline)) {
            const int s0 = kChunk * c + 1, row0 = dir ? Tb - 1 - s0 : s0;
            float res[kChunk], lf[kChunk];
            int ex[kChunk];
            // In the table the offset is that of the block's largest cell, to a binade, in every step, and no residual is above 0
            // (the gradients' rule on what their products hold counts on both): a step that kept its scale is moved by as many
            // binades as its largest cell lies beside the scale.  (What the blocks of this group read in LDS stays as it is.  With the
            // offsets as the walk has them, up to 44 binades above the largest cell, the backward at B = 16, L = 1024, T = 256 and
            // transition logits of standard deviation 3 and 5 sent steps to its direct form for nothing: 78.9 -> 68.2 and
            // 103.6 -> 93.6 us; the maxima cost the forward 0.7 us of 105 at L = 512, 1.1 of 57 in scoring.)
            int moved[kChunk] = {0, 0, 0, 0};
            if constexpr (!WIDE) {
                moved[0] = (__builtin_amdgcn_readlane(__builtin_bit_cast(int, kept), 31) >> 23) - (126 + kShift2);
                moved[2] = (__builtin_amdgcn_readlane(__builtin_bit_cast(int, kept), 63) >> 23) - (126 + kShift2);
            }
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {   // (a dead cell: log of the fraction 0)
                if constexpr (WIDE) {
                    ex[k] = __builtin_amdgcn_frexp_exp(v[k]) - CH::kShift;
                    lf[k] = fast_log2((float)__builtin_amdgcn_frexp_mant(v[k]));
                    res[k] = (float)(((double)ex[k] + (double)lf[k]) * 0.6931471805599453);
                } else {
                    ex[k] = __builtin_amdgcn_frexp_expf(v[k]) - kShift2;
                    lf[k] = fast_log2(__builtin_amdgcn_frexp_mantf(v[k]));
                    res[k] = ((float)(ex[k] - moved[k]) + lf[k]) * kLn2;
                }
            }
            const unsigned lane_off = (unsigned)(dir ? Lb - 1 - first - lane : first + lane) * 4u;
            char *row = const_cast<char *>(hat_c) + (unsigned)(row0 * L) * 4u;
            const int step = (dir ? -L : L) * 4;
            auto put = [&](const int k) __attribute__((always_inline)) {
                store_agent(reinterpret_cast<float *>(row + lane_off), res[k]);
                row += step;
            };
            const int steps = Tb - s0 < kChunk ? Tb - s0 : kChunk;
            if (__builtin_expect(steps == kChunk && first + kBlk <= Lb, 1)) { put(0); put(1); put(2); put(3); }
            else if (first + lane < Lb) { put(0); if (steps > 1) put(1); if (steps > 2) put(2); if (steps > 3) put(3); }
            const int k01 = lane & 1 ? kk[1] : kk[0], k23 = lane & 1 ? kk[3] : kk[2], kp = lane & 2 ? k23 : k01;
            const int kt = kp + (WIDE || (lane & 1) ? 0 : lane & 2 ? moved[2] : moved[0]);
            if (lane < steps)
                store_agent(reinterpret_cast<double *>(const_cast<char *>(off_c) + (unsigned)((dir ? row0 - lane : row0 + lane) * NBK + J) * 8u),
                            kt > kDeadBelow ? (double)kt * 0.6931471805599453 : (double)DAGX_NEG_INF);
            if (__builtin_expect(c == NC - 1 && J == NBb - 1, 0)) {   // the read-out
#pragma unroll
                for (int k = 0; k < kChunk; ++k)
                    if (k == steps - 1 && first + lane == Lb - 1) {
                        const double z = kk[k] > kDeadBelow ? ((double)(ex[k] + kk[k]) + (double)lf[k]) * 0.6931471805599453 : (double)DAGX_NEG_INF;
                        a.logz[slot * a.B + b] = z; if (slot == a.loss_dir) a.loss[b] = (float)z; store_agent(a.zfast + slot * a.B + b, z);
                    }
            }
            return kp;
        };
        for (int tau = first_stage; tau <= end_stage; ++tau) {
            const int par = tau & 1;
            // (per-lane addresses are formed anew in every stage: held across the loop they would cost the tiles their registers)
            const int lane = opaque_lane();
            // the foreign chunks this stage brings in: tau + 1 of the block below, which the walk of my first block wants, and
            // tau + 2 of the others, which the products of the next stage want
            const bool bring = FETCHES && f_blk[0] >= 0 && tau + 1 < NC;
            int published = 0;
            if (bring) published = load_agent(below);
            // The last two blocks' rows of the last stage are in memory when both their waves have come here, the other
            // blocks' of the stage before that (their waves have since waited for match rows requested behind them): the
            // second of the two publishes.  (In front of the walk, although it waits there: half way through it, where the rows are
            // there without a wait, B = 16, L = 1024, T = 64 takes 166 us instead of 158.)
            auto publish = [&]() __attribute__((always_inline)) {
                const int n = tau - (nblk - 1);                // chunks of the last block
                if (!producer || wave < nblk - 2 || n < 0 || n >= NC) return;
                wait_vmem_all();
                int both = 1;
                if (nblk > 1) {
                    if (lane == 0) both = __hip_atomic_fetch_add(published_by, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & 1;
                }
                if (lane == 0 && both) store_agent(prog + g, 2 + n);
            };
            // ---------------- walk my block through chunk tau - wave ----------------
            if (WALKS) {
                const int c = tau - wave;
                const bool more = c >= -1 && c + 1 < NC, live = c >= 0 && c < NC && c >= dest_lo(J) && c <= dest_hi(J);
                // what block J - 1 sends: its cells of this chunk
                const bool lower = live && J > 0 && c >= src_lo(J - 1) && c <= dest_hi(J - 1);
                Cell Ga[kChunk] = {0, 0, 0, 0};
                if (lower) {
                    __builtin_amdgcn_s_setprio(3);
                    const Cell *const src_cells = eb + ((own_src - 1) * D + slot_own) * 256;
                    if constexpr (WIDE) {
                        double out[4];
                        tile_product(t0, src_cells, lane, out);
                        double *const turn = reinterpret_cast<double *>(lds_raw + o.turn) + wave * 256;
#pragma unroll
                        for (int q = 0; q < 4; ++q) turn[(lane >> 4) * kBlk + 16 * q + (lane & 15)] = out[q];
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) Ga[k] = turn[k * kBlk + lane];
                    } else {
                        const f32x4 out = tile_product(t0, *reinterpret_cast<const f32x4 *>(src_cells + lane * 4));
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) Ga[k] = out[k];
                    }
                }
                publish();
                if (more) load_match(c + 1, lane);
                if (c >= 0 && c < NC) {
                    Cell *const cells = eb + own_src * D * 256 + cell_place<WIDE>(lane);
                    Cell *const cells_next = cells + next_slot(slot_own) * 256;
                    Cell *const cells_this = cells + slot_own * 256;
                    int kk[kChunk];
                    Cell v[kChunk];
                    if (live) {
                        __builtin_amdgcn_s_setprio(3);
                        // (lane <-> step) the exponents of what is sent; block J - 1's clamped as a tile's under the largest of the
                        // blocks below
                        const int rv = lds_i[o.part_scale + (wave * 2 + (par ^ 1)) * 4 + (lane & 3)];
                        int av = kDeadExp;
                        if (lower) {
                            av = lds_i[o.kap + ((own_src - 1) * D + slot_own) * 4 + (lane & 3)];
                            if (av - rv < CH::kFloor) av = upper ? rv + CH::kFloor : kDeadExp;
                        }
                        int A[kChunk], R[kChunk];
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) { A[k] = __builtin_amdgcn_readlane(av, k); R[k] = __builtin_amdgcn_readlane(rv, k); }
                        const Cell *const parts = part + (t.run_first * 2 + (par ^ 1)) * 256 + lane * (WIDE ? 1 : 4);
                        const float upper_half = lane >= 32 ? 1.f : 0.f;
                        Cell G[kChunk];
                        if constexpr (WIDE) {
#pragma unroll
                            for (int k = 0; k < kChunk; ++k) G[k] = parts[k * kBlk];
#pragma unroll 1
                            for (int u = 1; u < t.run_count; ++u)
#pragma unroll
                                for (int k = 0; k < kChunk; ++k) G[k] += parts[u * 512 + k * kBlk];
                        } else {
                            f32x4 sum = *reinterpret_cast<const f32x4 *>(parts);
                            if (t.run_count > 1) {
                                f32x4 sum1 = *reinterpret_cast<const f32x4 *>(parts + 512);
                                if (t.run_count > 2) {
                                    sum += *reinterpret_cast<const f32x4 *>(parts + 1024);
#pragma unroll 1
                                    for (int u = 3; u < t.run_count; ++u) sum += *reinterpret_cast<const f32x4 *>(parts + u * 512);
                                }
                                sum += sum1;
                            }
#pragma unroll
                            for (int k = 0; k < kChunk; ++k) G[k] = sum[k];
                        }
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            // (float32, kSpare: every other step does not scale its cells by their largest)
                            const int most = A[k] > R[k] ? A[k] : R[k], ref = (kap > most ? kap : most) + (WIDE || (k & 1) ? 0 : kSpare);
                            // (what ldexp flushes of either part is under flush_up, too)
                            const Cell x = (pow2(triangle_dot(t2, e, upper_half), kap - ref) + flush_up) + (pow2(G[k], R[k] - ref) + pow2(Ga[k], A[k] - ref));
                            // (upper sweep: a cell never flushes, live or not -- what a dead one gets is of the size of what is flushed.
                            //  So the scale must not be applied to the finished product x exp(match), which may have flushed: it is
                            //  split between the factors, or, in float64, joined with the match exponent.)
                            if constexpr (WIDE) {
                                const double y = x * (double)mt[k];
                                // exponent of y 2^mt_exp; a cell of 0 has the least (exp(match) is 0) or no weight (lower sweep)
                                const int tb = wave64_max_int((int)((unsigned)(__builtin_bit_cast(unsigned long long, y) >> 52)) + mt_exp[k]);
                                kap = __builtin_amdgcn_ballot_w64(y != 0.0) != 0 ? tb + ref + N[k] - (1022 + CH::kShift + CH::kLinkShift) : kDeadExp;
                                e = pow2(y, mt_exp[k] + (1022 + CH::kShift) - tb) + tiny_up;
                            } else {
                                const float y = x * mt[k];
                                auto scaled = [&](const int base) __attribute__((always_inline)) {
                                    // the exponent of the largest cell, at least that of 2^-72: its reciprocal has to be a float32 number
                                    const unsigned top = wave64_max_positive(y);
                                    const int tb = (int)(top >> 23) > 55 ? (int)(top >> 23) : 55, up = 253 + kShift2 - tb;
                                    kap = top ? base + tb : kDeadExp;
                                    // (a factor below 1 goes to x, one above 1 to exp(match), which is 0 or at least 2^-126)
                                    e = __builtin_fmaf(x * __builtin_bit_cast(float, (unsigned)(up < 127 ? up : 127) << 23),
                                                       mt[k] * __builtin_bit_cast(float, (unsigned)(up > 127 ? up : 127) << 23), tiny_up);
                                };
                                if (k & 1) scaled(ref + N[k] - (126 + 2 * kShift2));
                                else {   // at most 2^60, and mostly 15 to 45 binades lower
                                    kap = ref + N[k] - kShift2;
                                    if (__builtin_expect(__builtin_amdgcn_ballot_w64(y >= kScaleBelow) != 0, 1)) e = y + tiny_up;
                                    else scaled(kap - (126 + kShift2));   // (so far below that it would cost the cells under it their range)
                                }
                            }
                            kk[k] = kap;
                            v[k] = e;
                            if (k < kChunk - 1) cells_this[CH::kStepPitch * (k + 1)] = e; else cells_next[0] = e;
                        }
                        __builtin_amdgcn_s_setprio(0);
                    } else {
                        e = 0; kap = kDeadExp;
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            kk[k] = kDeadExp;
                            v[k] = 0;
                            if (k < kChunk - 1) cells_this[CH::kStepPitch * (k + 1)] = 0; else cells_next[0] = 0;
                        }
                    }
                    float kept = 0.f;
                    if constexpr (!WIDE) kept = fold_two(v[0], v[2]);
                    if (more) convert_match(c + 1, lane, std::bool_constant<!WIDE>{}, kept);   // (in front of the stores: what it waits for is older than they)
                    else {
                        if constexpr (!WIDE) half_max(kept);
                        wait_vmem_all();
                    }
                    const int kp = write_out(c, v, kk, kept, lane);
                    const int sl = (lane & 3) < kChunk - 1 ? slot_own * 4 + 1 + (lane & 3) : next_slot(slot_own) * 4;
                    if (lane < kChunk) lds_i[o.kap + own_src * D * 4 + sl] = kp;
                    slot_own = next_slot(slot_own);
                }
                else if (more) { float none = 0.f; convert_match(c + 1, lane, std::false_type{}, none); }
                else if (c == NC) wait_vmem_all();
            }
            // ---------------- multiply out what my tiles' blocks (q of the group) receive in chunk tau + 1 - q ----------------
            if (t.count > 0) {
                // (float32: the LDS reads of two tiles are requested before the first is waited for, the third's behind the first)
                f32x4 ev[2];
                int kv[kTilesPerWave], rv[kTilesPerWave], at[kTilesPerWave];
                bool go[kTilesPerWave], src[kTilesPerWave];
                const int step = WIDE ? lane >> 4 : lane & 3, other = WIDE ? lane & 15 : lane >> 2;   // (lane <-> step and block of what leads here)
                auto cells_of = [&](const int u) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4 *>(lds_raw + o.eb + at[u] + lane * 4); };
#pragma unroll
                for (int u = WALKS ? 1 : 0; u < (WALKS ? 2 : kTilesPerWave); ++u) {
                    go[u] = tau >= t_from[u] && tau <= t_to[u];
                    src[u] = tau >= t_src_from[u] && tau <= t_src_to[u];
                    if (go[u]) {
                        int sl = ring + t_shift[u]; sl -= sl >= D ? D : 0;
                        at[u] = t_cells[u] + sl * 256;
                        if (!WIDE && u < 2) ev[u] = cells_of(u);
                        kv[u] = lds_i[t_kaps[u] + sl * 4 + step];
                        if (t.start[u]) {
                            const int n = other < t_scales[u] ? other : 0;
                            rv[u] = lds_i[t_scale_at[u] + sl * 4 + n * (D * 4) + step];
                        }
                    }
                }
                Cell G[4] = {0, 0, 0, 0};
                int R = kDeadExp;
                auto product = [&](const int u, const Tile &tile) __attribute__((always_inline)) {
                    if (!go[u]) return;
                    if (t.start[u]) {   // the scale: the largest exponent, step by step, among all blocks that lead here
                        if constexpr (WIDE) R = row16_max_int(rv[u]); else R = by_step_max(rv[u]);
#pragma unroll
                        for (int k = 0; k < 4; ++k) G[k] = 0;
                    }
                    if (src[u]) {
                        if constexpr (WIDE) {
                            double v[4];
                            tile_product(tile, eb + at[u], lane, v);
                            const double f = pow2_clamped_wide(kv[u] - R, floor_exp);
#pragma unroll
                            for (int k = 0; k < 4; ++k) G[k] = __builtin_fma(v[k], f, G[k]);
                        } else {
                            const f32x4 v = tile_product(tile, ev[u & 1]);
                            f32x4 sum = {G[0], G[1], G[2], G[3]};
                            scaled4(sum, pow2_clamped(kv[u] - R, floor_exp), v);
#pragma unroll
                            for (int k = 0; k < 4; ++k) G[k] = sum[k];
                        }
                    }
                    if (t.end[u]) {
                        Cell *const to = part + (t.run[u] * 2 + par) * 256;
                        if constexpr (WIDE) {
#pragma unroll
                            for (int k = 0; k < 4; ++k) to[(lane >> 4) * kBlk + 16 * k + (lane & 15)] = G[k];
                            if (t.lead[u] && (lane & 15) == 0) lds_i[o.part_scale + (t.q[u] * 2 + par) * 4 + step] = R;
                        } else {
                            *reinterpret_cast<f32x4 *>(to + lane * 4) = f32x4{G[0], G[1], G[2], G[3]};
                            if (t.lead[u] && lane < 4) lds_i[o.part_scale + (t.q[u] * 2 + par) * 4 + lane] = R;
                        }
                    }
                };
                if (!WALKS) product(0, t0);
                if (!WIDE && !WALKS && go[2]) ev[0] = cells_of(2);
                product(1, t1);
                if (!WALKS) product(2, t2);
            }
            // ---------------- table rows of foreign blocks: requested a stage ago if they were published by then ----------------
            if (bring) {
                published = __builtin_amdgcn_readfirstlane(published);
                if (published > seen) seen = published;
                auto chunk_of = [&](const int u, const int stage) { return stage + (f_blk[u] == jb0 - 1 ? 1 : 2); };
                auto request = [&](const int stage) __attribute__((always_inline)) {   // what a stage brings in
#pragma unroll
                    for (int u = 0; u < kForeign; ++u) {
                        if (f_blk[u] < 0) break;
                        const int c = chunk_of(u, stage);
                        if (c >= 0 && c < NC) request_rows(f_blk[u], c, lane);
                    }
                    requested = stage;
                };
                if (requested < tau) {
                    int spins = 0;
                    while (seen < tau + 4) {
                        __builtin_amdgcn_s_sleep(1);
                        seen = __builtin_amdgcn_readfirstlane(load_agent(below));
                        if (++spins > kSpinLimit) { *s_abort_p = 1; break; }
                    }
                    if (seen >= tau + 4) request(tau);
                }
                wait_vmem_all();
#pragma unroll
                for (int u = 0; u < kForeign; ++u) {
                    if (f_blk[u] < 0) break;
                    const int c = chunk_of(u, tau);
                    int sl = ring + c - tau; sl -= sl >= D ? D : 0;
                    if (c >= 0 && c < NC) convert_rows(f_blk[u], sl, lane);
                }
                if (tau + 2 < NC && seen >= tau + 5) request(tau + 1);
            }
            ring = next_slot(ring);
            __syncthreads();
            if (consumer && __builtin_amdgcn_readfirstlane(*s_abort_p)) return;
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
    if (consumer && __builtin_amdgcn_readfirstlane(*s_abort_p)) {   // a producer never showed up: hand the sample on and let consumers go on
        wait_vmem_all();
        if (tid == 0) { store_agent(risk, 1); store_agent(prog + g, 1 << 30); }
    }
}

// The two read-outs of a sample's tile sweeps bracket log Z: one sweep rounds everything the linear domain
// cannot hold down to 0, the other up to the smallest number it holds.  Where they agree, what was flushed carried
// no mass that matters and either read-out is log Z to the tolerance; where they do not (or one is not finite,
// or a NaN) the sample is done again: by the wide sweeps, then by the log-domain kernel.  The tolerance bounds the
// mass the upper sweep has rounded up, which the gradients would see as posteriors of that size where the true ones
// are 0: 5e-5, half of what the gradients are held to.  On top of it comes what rounding alone leaves between two
// sweeps.  The float32 sweeps carry cell values as float32 numbers relative to a float64 reference: measured between
// an alpha and a beta sweep up to 1.5e-5 at |log Z| = 800 on benign inputs and 3e-5 ... 5e-5 at 2600 ... 3500, hence
// the term 1e-7 |Z|; but never more than 1e-4, what the gradients are held to, however large |log Z| (the few
// samples of long, peaked graphs whose read-outs differ by more through rounding alone cost a pass of the wide
// sweeps).  The wide sweeps carry them as float64 numbers whose
// logarithm comes from v_log_f32 of a fraction in [1/2, 1), 1e-7 absolute per step: 1e-8 |Z| covers it.  (With
// float32 cell values the wide sweeps needed 2e-4 + 2e-7 |Z|, and that passed upper sweeps that had rounded
// 3e-4 ... 6e-4 of mass up: their transitions are clamped at exp(-175) times the scale, which is not nothing when
// the path that carries the mass lies as deep.)
__device__ __forceinline__ bool readouts_disagree(double za, double zb, bool wide) {
    if (!(za > (double)DAGX_NEG_INF) || !(zb > (double)DAGX_NEG_INF) || za != za || zb != zb) return true;
    return !(fabs(za - zb) <= (wide ? 1e-8 * fabs(zb) + 5e-5 : fmin(1e-7 * fabs(zb) + 5e-5, 1e-4)));
}

template <typename TM, typename TL, bool WIDE>
__global__ __launch_bounds__(kTileWaves * kWave) void dag_sweep_tiles_kernel(TileSweepArgs a) {
    extern __shared__ __align__(16) float lds_raw[];
    __shared__ int gstart[kTileCap + 2];
    __shared__ int s_ticket, s_abort;
    const int tid = threadIdx.x;
    const int C = a.C;
    // The wide launch behind a float32 launch that flagged nothing (the usual case) ends here, after one load: the
    // float32 launch counts the samples it flags in word 2 of the pipeline words, the wide launch clears it.
    if constexpr (WIDE) { if (a.sync[2] == 0) return; }
    // (all that the ticket waits for in one round trip to the argument block)
    int *sync = a.sync;
    int ntable = a.choice.ntable, least = a.choice.least, B = a.B, ndir = a.ndir;
    asm volatile("" : "+s"(sync), "+s"(ntable), "+s"(least), "+s"(B), "+s"(ndir));
    const int B8 = (B + 7) & ~7;
    // Which table, and with it how many workgroups take part: all of them come to the same answer from the lengths alone.  The
    // others leave at once; they are the last of the grid, so they cost a CU that has become free a look at the lengths.
    int mine = 0, used = 0, workgroups = ndir * B8 * least;   // (lane <-> sample) groups of a sample, table
    if (__builtin_expect(ntable > 1, 0)) {   // (unlikely: out of the way of batches without a choice, which else wait for these instructions:
                                             //  scoring at B = 40, L = 328 58.6 us for 57.5)
        const int lane = tid & (kWave - 1);
        const int64_t len = a.out_len[lane < B ? lane : 0];
        const int nb = len >= 1 && len <= a.L ? ((int)len + kBlk - 1) / kBlk : 1;
        for (int x = ntable - 1; x > 0 && used == 0; --x) {
            const int n = lane < B ? (int)(a.choice.ngroups[x] >> (4 * (nb - 1))) & 15 : 0;
            int all = n;
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) all += __shfl_xor(all, d, kWave);
            all = __builtin_amdgcn_readfirstlane(all) * ndir;
            if (all <= kSweepCus) { mine = n; used = x; workgroups = all; }
        }
        used = __builtin_amdgcn_readfirstlane(used);
        workgroups = __builtin_amdgcn_readfirstlane(workgroups);
        if ((int)blockIdx.x >= workgroups) return;
    }
    if (tid == 0) { s_ticket = atomicAdd(sync, 1); s_abort = 0; }
    __syncthreads();
    // ticket -> (group, sweep, sample): first group 0 of every sweep of every sample, then every group 1, and so on.
    // Every group waits only on groups with a smaller ticket, so a waiting workgroup's producers have already
    // started; and the workgroups that the dispatcher reaches last (it needs several microseconds for the grid)
    // are consumers, which could not start any sooner than their producers' first rows anyway.  The two sweeps of a
    // sample are 8 tickets apart, the workgroups of a sample a multiple of 8 (table 0): they share an XCD and its L2.
    const int k = __builtin_amdgcn_readfirstlane(s_ticket);
    int g, b_k, slot_k, groups = least;
    bool has_sample;
    if (__builtin_expect(used == 0, 1)) {
        const int runs = ndir * (B8 / 8);   // runs of eight (sweep, sample) pairs
        const int run = (k / 8) % runs;
        g = k / (8 * runs); slot_k = run % ndir;
        b_k = (run / ndir) * 8 + (k % 8);
        has_sample = g < least && b_k < B;
    } else {   // samples without a group g are passed over; k < workgroups, so there is a (group, sweep, sample) for it
        int r = k, n = 0;
        unsigned long long have = 0;
#pragma unroll 1
        for (g = 0; g < C; ++g) {
            have = __builtin_amdgcn_ballot_w64(mine > g);
            n = __builtin_popcountll(have);
            if (r < ndir * n) break;
            r -= ndir * n;
        }
        int rank;
        place_of_ticket(r, n, ndir, rank, slot_k);
        const int lane = tid & (kWave - 1);
        const int before = __builtin_popcountll(have & ((1ull << lane) - 1));
        const unsigned long long at = __builtin_amdgcn_ballot_w64((have >> lane & 1) != 0 && before == rank);
        has_sample = g < C && at != 0;
        b_k = has_sample ? (int)__builtin_ctzll(at) : 0;
        groups = __builtin_amdgcn_readlane(mine, b_k);
    }
    has_sample = __builtin_amdgcn_readfirstlane(has_sample) != 0;
    g = __builtin_amdgcn_readfirstlane(g);
    const int b = __builtin_amdgcn_readfirstlane(has_sample ? b_k : 0), slot = __builtin_amdgcn_readfirstlane(has_sample ? slot_k : 0);
    // a launch for flagged samples only (the wide variant behind the float32 one): the workgroups of the others
    // leave at once, through the same bookkeeping
    const bool skip = has_sample && a.only_flagged && a.flags[b] != 1;
    if (has_sample && !skip) {
        sweep_chunks_group<TM, TL, WIDE>(a, a.table[used], b, slot, g, lds_raw, gstart, &s_abort);
    }
    // ---- leaving ----
    wait_vmem_all();   // this wave's stores (table rows, read-outs) are complete
    __syncthreads();
    if (tid == 0) {
        if (has_sample) {
            int *left = a.sync + 16 + a.ndir * a.B * C + b, *risk = left + a.B;
            const int n = __hip_atomic_fetch_add(left, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
            if (n == a.ndir * groups) {   // every workgroup of the sample has left
                bool bad = load_agent(risk) != 0;
                const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
                if (!bad && lengths_ok(Lb, Tb, a.L, a.T)) {
                    bad = readouts_disagree(load_agent(a.zfast + b), load_agent(a.zfast + a.B + b), WIDE);
                }
                if (!skip) a.flags[b] = bad ? 1 : (WIDE ? 2 : 0);   // 1: still to be done; 2: settled by the wide variant
                if (!WIDE && bad) __hip_atomic_fetch_add(a.sync + 2, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (int d = 0; d < a.ndir; ++d)
                    for (int q = 0; q < C; ++q) store_agent(a.sync + 16 + (d * a.B + b) * C + q, 0);
                store_agent(left, 0);
                store_agent(risk, 0);
                for (int d = 0; d < a.ndir; ++d) store_agent(a.zfast + d * a.B + b, 0.0);
            }
        }
        const int n_all = __hip_atomic_fetch_add(a.sync + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
        if (n_all == workgroups) { store_agent(a.sync, 0); store_agent(a.sync + 1, 0); if (WIDE) store_agent(a.sync + 2, 0); }
    }
}

// In front of a forward that starts with the float64 sweeps: every sample marked "still to be done", and the count the
// float32 launch would have left, so that the float64 launch does not take itself for idle.
__global__ void dag_mark_all_kernel(int *flags, int B, int *sync) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < B) flags[i] = 1;
    if (i == 0) store_agent(sync + 2, B);
}

__global__ void dag_fill_int_kernel(int *p, int n, int v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ================================================================================================
// Gradients
// ================================================================================================

__device__ __forceinline__ bool finite_d(double z) { return z > (double)DAGX_NEG_INF && z < (double)__builtin_huge_valf(); }

// Clearing the part of grad_links that the tile kernel does not write.  Per sample:
//   - valid lengths, T_b >= 2, finite Z: the tile kernel writes the entries with i + d + 1 < L_b, so row i
//     is cleared from d = max(0, L_b - 1 - i) on;
//   - otherwise the gradient is zero everywhere and the whole sample is cleared.
// A workgroup of four waves owns `rows` consecutive rows of one sample, a wave clears a row at a time:
// 16-byte stores between element-wise head and tail (row starts are only element-aligned).
typedef uint32_t fill_u32x4 __attribute__((ext_vector_type(4)));
struct ZeroJob {
    unsigned char *base; int elem;       // grad_links and its element size (2 or 4)
    const int64_t *out_len, *tgt_len; const double *logz;   // logz: [2][B], the second row is Z
    int B, T, L, translen;
    int rows, chunks;                    // rows per workgroup, workgroups per sample
    int blocks;                          // B * chunks; 0: nothing to clear
};
__device__ __forceinline__ void zero_elem(unsigned char *p, int elem) {
    if (elem == 4) *reinterpret_cast<uint32_t *>(p) = 0u; else *reinterpret_cast<uint16_t *>(p) = 0;
}
__device__ __forceinline__ void zero_part(const ZeroJob &z, int block) {
    const int tid = threadIdx.x;
    const int b = block / z.chunks, chunk = block % z.chunks;
    const int Lb = (int)z.out_len[b], Tb = (int)z.tgt_len[b];
    const double Z = z.logz[z.B + b];
    const bool tiled = lengths_ok(Lb, Tb, z.L, z.T) && Tb >= 2 && finite_d(Z);
    const int i_end = (chunk + 1) * z.rows < z.L ? (chunk + 1) * z.rows : z.L;
    const int lane = tid & (kWave - 1);
    for (int i = chunk * z.rows + (tid >> 6); i < i_end; i += (int)(blockDim.x >> 6)) {   // one wave per row
        int d0 = tiled ? Lb - 1 - i : 0;
        if (d0 < 0) d0 = 0;
        if (d0 >= z.translen) continue;
        unsigned char *row = z.base + ((int64_t)b * z.L + i) * z.translen * z.elem;
        const unsigned misalign = (unsigned)(reinterpret_cast<uintptr_t>(row) & 15u);
        const unsigned s = (unsigned)(d0 * z.elem), e = (unsigned)(z.translen * z.elem);   // byte range [s, e) of the row
        unsigned body = ((s + misalign + 15u) & ~15u) - misalign; if (body > e) body = e;  // first 16-byte boundary at or after s
        const unsigned body_end = body + ((e - body) & ~15u);
        for (unsigned o = s + lane * z.elem; o < body; o += kWave * z.elem) zero_elem(row + o, z.elem);
        for (unsigned o = body + lane * 16u; o < body_end; o += kWave * 16u) *reinterpret_cast<fill_u32x4 *>(row + o) = fill_u32x4{0u, 0u, 0u, 0u};
        for (unsigned o = body_end + lane * z.elem; o < e; o += kWave * z.elem) zero_elem(row + o, z.elem);
    }
}

// grad_match[b][t][j] = g_b * exp(alpha + beta - match - Z), Z = beta read-out; 0 outside the sample,
// where match is +-inf, or when Z is not finite.  The first zero.blocks workgroups of the launch clear
// the grad_links buffer instead (one launch less in front of the tile kernel).
template <typename TM>
__device__ __forceinline__ void grad_match_cell(
    const float *__restrict__ grad_out, int64_t gstride, const float *__restrict__ ahat, const float *__restrict__ bhat,
    const double *__restrict__ aoff, const double *__restrict__ boff, const double *__restrict__ logz,
    const TM *__restrict__ match, int64_t ms0, int64_t ms1, int64_t ms2,
    const int64_t *__restrict__ out_len, const int64_t *__restrict__ tgt_len, int B, int T, int L, int NBK,
    TM *__restrict__ grad_match, int b, int t, int j) {
    if (j >= L) return;
    const int Lb = (int)out_len[b], Tb = (int)tgt_len[b];
    const int64_t o = ((int64_t)b * T + t) * L + j;
    float r = 0.f;
    if (lengths_ok(Lb, Tb, L, T) && t < Tb && j < Lb) {
        const double Z = logz[B + b];
        const float m = to_float(match[b * ms0 + t * ms1 + j * ms2]);
        if (finite_d(Z) && m > DAGX_NEG_INF && m < __builtin_huge_valf()) {
            const int64_t ob = ((int64_t)b * T + t) * NBK;
            const double k = aoff[ob + j / kBlk] + boff[ob + (Lb - 1 - j) / kBlk] - Z;  // -inf if a block is dead
            // (summed in float64: with token log-probabilities a hundred nats apart the four terms are hundreds each and
            //  cancel, and float32 sums of them are off by 1e-4 of a posterior near 1)
            const float x = (float)((((double)ahat[o] + (double)bhat[o]) + k) - (double)m);
            r = grad_out[b * gstride] * fast_exp2(x * kLog2e);
        }
    }
    grad_match[o] = from_float<TM>(r);
}
template <typename TM>
__global__ __launch_bounds__(256) void dag_grad_match_kernel(
    const float *__restrict__ grad_out, int64_t gstride, const float *__restrict__ ahat, const float *__restrict__ bhat,
    const double *__restrict__ aoff, const double *__restrict__ boff, const double *__restrict__ logz,
    const TM *__restrict__ match, int64_t ms0, int64_t ms1, int64_t ms2,
    const int64_t *__restrict__ out_len, const int64_t *__restrict__ tgt_len, int B, int T, int L, int NBK,
    TM *__restrict__ grad_match, ZeroJob zero) {
    if ((int)blockIdx.x < zero.blocks) { zero_part(zero, blockIdx.x); return; }
    const int id = blockIdx.x - zero.blocks, nx = (L + 255) / 256;
    grad_match_cell<TM>(grad_out, gstride, ahat, bhat, aoff, boff, logz, match, ms0, ms1, ms2, out_len, tgt_len, B, T, L, NBK,
                        grad_match, id / (nx * T), (id / nx) % T, (id % nx) * 256 + (int)threadIdx.x);
}

// grad_links[b][i][d] = g_b * sum_{t=0}^{T_b-2} exp(alpha[t][i] + E[i][d] + beta[t+1][i+d+1] - Z), direct form
// (each term <= 1), for graphs the tile kernel does not take (L > 1024) and for the log-domain-only mode.
// Tile: RI rows x 64 transitions per workgroup.  The steps are walked in chunks of kDirectSteps: per chunk
// the alpha residuals of the rows (float32) and, per column, the beta residual plus every block offset of the
// step minus Z (float64: the offsets are large and cancel) are staged in LDS; a term is
// exp(float32(float64 sum) + E).
constexpr int kDirectSteps = 32;
template <typename TL, int RI>
__global__ __launch_bounds__(256) void dag_grad_links_kernel(
    const float *__restrict__ grad_out, int64_t gstride, const float *__restrict__ ahat, const float *__restrict__ bhat,
    const double *__restrict__ aoff, const double *__restrict__ boff, const double *__restrict__ logz,
    const TL *__restrict__ links, const int64_t *__restrict__ out_len, const int64_t *__restrict__ tgt_len,
    int B, int T, int L, int translen, int NBK, TL *__restrict__ grad_links) {
    constexpr int JW = 64 + RI;          // columns of beta touched by the tile (j = i+d+1)
    __shared__ float a_s[kDirectSteps][RI];     // alpha_hat[t][i]
    __shared__ double b_s[kDirectSteps][JW];    // beta_hat[t+1][j] + beta_off[t+1][blk(j)] + alpha_off[t][blk(i0)] - Z
    const int b = blockIdx.z;
    const int d0 = blockIdx.x * 64;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int Lb = (int)out_len[b], Tb = (int)tgt_len[b];
    TL *gl = grad_links + (int64_t)b * L * translen;
    const int d = d0 + lane;
    const bool ok = lengths_ok(Lb, Tb, L, T);
    const double Z = ok ? logz[B + b] : (double)DAGX_NEG_INF;
    const float g = grad_out[b * gstride];
    const float *al = ahat + (int64_t)b * T * L, *be = bhat + (int64_t)b * T * L;
    const double *ao = aoff + (int64_t)b * T * NBK, *bo = boff + (int64_t)b * T * NBK;
    // a workgroup walks the row tiles blockIdx.y, blockIdx.y + gridDim.y, ... of its column strip
    for (int i0 = blockIdx.y * RI; i0 < L; i0 += gridDim.y * RI) {
        const bool live = ok && finite_d(Z) && i0 < Lb - 1 && i0 + d0 + 1 < Lb && Tb >= 2;
        if (!live) {  // whole tile is zero
            for (int r = w; r < RI; r += 4) {
                const int i = i0 + r;
                if (i < L && d < translen) gl[(int64_t)i * translen + d] = from_float<TL>(0.f);
            }
            continue;
        }
        const int slack = Lb - Tb;
        const int jbase = i0 + d0 + 1;
        // useful steps for this tile: t in [tlo, thi]
        int tlo = jbase - 1 - slack; if (tlo < 0) tlo = 0;
        int thi = i0 + RI - 1; if (thi > Tb - 2) thi = Tb - 2;
        const int ablk0 = i0 / kBlk;         // RI divides 64: the rows of a tile share one alpha block
        float e[RI / 4], acc[RI / 4];
#pragma unroll
        for (int q = 0; q < RI / 4; ++q) {
            const int i = i0 + w + 4 * q, j = i + d + 1;
            acc[q] = 0.f;
            e[q] = (i < Lb - 1 && j < Lb && d < translen) ? to_float(links[((int64_t)b * L + i) * translen + d]) : DAGX_NEG_INF;
        }
        for (int c0 = tlo; c0 <= thi; c0 += kDirectSteps) {
            const int nt = thi - c0 + 1 < kDirectSteps ? thi - c0 + 1 : kDirectSteps;
            __syncthreads();   // the previous chunk's (or tile's) reads of the staged arrays are done
            for (int k = tid; k < nt * RI; k += 256) {
                const int t = c0 + k / RI, r = k % RI, i = i0 + r;
                a_s[k / RI][r] = i < Lb ? al[(int64_t)t * L + i] : DAGX_NEG_INF;
            }
            for (int k = tid; k < nt * JW; k += 256) {
                const int t = c0 + k / JW, c = k % JW, j = jbase + c;
                double v = (double)DAGX_NEG_INF;
                if (j < Lb) {
                    const double ka = ao[(int64_t)t * NBK + ablk0], kb = bo[(int64_t)(t + 1) * NBK + (Lb - 1 - j) / kBlk];
                    if (ka > (double)DAGX_NEG_INF && kb > (double)DAGX_NEG_INF)
                        v = (double)be[(int64_t)(t + 1) * L + j] + ((ka - Z) + kb);
                }
                b_s[k / JW][c] = v;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < RI / 4; ++q) {
                const int r = w + 4 * q;
                if (e[q] > DAGX_NEG_INF) {
                    const int c = r + lane;      // j - jbase
                    float sum = 0.f;
                    for (int k = 0; k < nt; ++k) {
                        const float x = (float)(b_s[k][c] + (double)a_s[k][r]) + e[q];
                        sum += fast_exp2(x * kLog2e);
                    }
                    acc[q] += sum;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < RI / 4; ++q) {
            const int i = i0 + w + 4 * q;
            if (i < L && d < translen) gl[(int64_t)i * translen + d] = from_float<TL>(g * acc[q]);
        }
    }   // row tiles
}

// ------------------------------------------------------------------------------------------------
// grad_links, block-scaled form.  With ea = exp(alpha_hat), eb = exp(beta_hat) (both in [0,1]) and
// the per-step factor K_t = exp(alpha_off[t][blk(i)] + beta_off[t+1][blk(j)] - Z),
//     grad_links[i][j] = g * P[i][j] * sum_t (K_t^(1/2) ea[t][i]) * (K_t^(1/2) eb[t+1][j]),
// a matrix product over the steps, in fp32 on the matrix cores.  One wave per 32-row x 64-column
// tile: two 32x32 accumulator blocks, v_mfma_f32_32x32x2_f32 consuming two steps at a time.  Its
// operand layout (lane = 32 * k + row of A / column of B) is exactly what a coalesced load of two
// table rows gives, so the factors go from global memory through one exponential straight into the
// MFMA.  The per-step scale factors sit in a small LDS table, one read per operand and step pair.
//
// When the factored form is safe.  A term exp(alpha[t][i] + E + beta[t+1][j] - Z) is at most 1; its two
// factors are formed separately, and one of them can leave the float32 range although the term does not.
// With x_t = log K_t for the largest blocks of the tile, each factor carries half of it: a factor can only
// flush when its residual is below -87 - x_t / 2, and then every term it belongs to is below
// exp(x_t / 2 - 87) (the other residual and E are <= 0).  And a cell's sum over n steps is at most n exp(max x_t)
// (the residuals are <= 0), whatever its transition.  So the matrix product takes the steps with
// x_t <= 88 - log(n), n = the steps of the tile: their sums cannot leave float32 (its largest number is exp(88.7))
// and what the factored form loses of them is below exp(-43) per term.  The other steps of the tile (inputs whose
// posterior sits far under the block maxima: sharply peaked transitions, pinned nodes) are left out of the product
// (their scale entries are -inf) and added afterwards, by the same wave, in the direct form: every term from a
// float64 sum of its parts, the transition inside the exponent.  A sum that is not finite all the same (a NaN in
// the tables) sends the whole tile through the direct form.  All in the same launch, with no check afterwards and
// no second kernel.  (A looser bound for the product, 120, with a check of the sums and a second product under the
// tight bound where one overflowed, keeps moderately peaked inputs off the direct steps -- 0.036 against 0.048 ms
// for the x10 test batch -- but the second copy of the loop costs every tile 7 % through the register allocation.)
// ------------------------------------------------------------------------------------------------

typedef float f32x16 __attribute__((ext_vector_type(16)));
// log K_t up to which a step of a tile of n steps goes through the matrix product
__device__ __forceinline__ double safe_log_k(int n) { return (double)(88.0f - fast_log2((float)(n > 1 ? n : 1)) * kLn2); }

struct GradTileArgs {
    const float *grad_out; int64_t gstride;
    const float *ahat, *bhat; const double *aoff, *boff, *logz;
    const void *links; void *grad_links;
    const int64_t *out_len, *tgt_len;
    int B, T, L, translen, NBK;
    int ntile;                           // live (row block, column block) pairs of a full-length sample
    unsigned char tile_bi[kMaxBlocksFast * (kMaxBlocksFast + 1) / 2], tile_jt[kMaxBlocksFast * (kMaxBlocksFast + 1) / 2];
    // Work that rides in the same launch, behind the tile workgroups (which start first and are bound by
    // their chains of memory round trips, so that these streaming workgroups fill the machine around them):
    // the clearing of the part of grad_links no tile writes, and grad_match (four 64-cell pieces of a table
    // row per workgroup).  tile_blocks = 2 * ntile * B; then zero.blocks, then match_blocks.
    int tile_blocks, match_blocks;
    ZeroJob zero;
    const void *match; int match_dtype; int64_t ms0, ms1, ms2; void *grad_match;
};
// Four cells of grad_match per lane (one step t of one sample, 256 consecutive positions per wave): the same values
// as grad_match_cell, but every load is requested up front, without conditions (indices clamped into the tables; what
// must not count is masked at the end), so that a wave waits for two memory round trips (the sample's lengths, which
// the beta offsets' index needs, then everything else) instead of three per cell.  These workgroups ride in the
// slots the gradient tiles leave free, a few hundred at a time: what they cost is their latency.
template <typename TM>
__device__ __forceinline__ void grad_match_cells4(const GradTileArgs &a, const TM *__restrict__ match, TM *__restrict__ grad_match,
                                                   const int b, const int t, const int j0) {
    const int L = a.L, T = a.T, NBK = a.NBK;
    const int64_t row = ((int64_t)b * T + t) * L, ob = ((int64_t)b * T + t) * NBK;
    float m[4], ah[4], bh[4];
    double ao[4];
    int jc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int j = j0 + u * kWave;
        jc[u] = j < L ? j : L - 1;
        m[u] = to_float(match[b * a.ms0 + t * a.ms1 + jc[u] * a.ms2]);
        ah[u] = a.ahat[row + jc[u]];
        bh[u] = a.bhat[row + jc[u]];
        ao[u] = a.aoff[ob + jc[u] / kBlk];
    }
    const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
    const double Z = a.logz[a.B + b];
    const float g = a.grad_out[b * a.gstride];
    const bool sample_ok = lengths_ok(Lb, Tb, L, T) && t < Tb && finite_d(Z);
    double bo[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        int q = (Lb - 1 - jc[u]) / kBlk;
        q = q < 0 ? 0 : (q < NBK ? q : NBK - 1);
        bo[u] = a.boff[ob + q];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int j = j0 + u * kWave;
        float r = 0.f;
        if (sample_ok && j < Lb && m[u] > DAGX_NEG_INF && m[u] < __builtin_huge_valf()) {
            const double k = ao[u] + bo[u] - Z;  // -inf if a block is dead
            const float x = (float)((((double)ah[u] + (double)bh[u]) + k) - (double)m[u]);   // (float64: see grad_match_cell)
            r = g * fast_exp2(x * kLog2e);
        }
        if (j < L) grad_match[row + j] = from_float<TM>(r);
    }
}

__device__ __forceinline__ void grad_side_jobs(const GradTileArgs &a, int id) {
    if (id < a.zero.blocks) { zero_part(a.zero, id); return; }
    id -= a.zero.blocks;
    const int nx = (a.L + 255) / 256;
    const int b = id / (nx * a.T), t = (id / nx) % a.T, j0 = (id % nx) * 256 + (int)threadIdx.x;
    switch (a.match_dtype) {
        case DAGX_F32: grad_match_cells4<float>(a, static_cast<const float *>(a.match), static_cast<float *>(a.grad_match), b, t, j0); break;
        case DAGX_F16: grad_match_cells4<__half>(a, static_cast<const __half *>(a.match), static_cast<__half *>(a.grad_match), b, t, j0); break;
        default: grad_match_cells4<bf16_t>(a, static_cast<const bf16_t *>(a.match), static_cast<bf16_t *>(a.grad_match), b, t, j0); break;
    }
}

// The direct form of one 32 x 64 tile, computed by one wave (see above for when).  Lane (half, l32)
// owns the columns j0 + l32 and j0 + 32 + l32 and the rows i0 + 8 q + 4 half + m (q, m < 4): cell (jh, v) of a
// lane is exp(float32(float64(beta side of its column) + float64(alpha residual of its row)) + E), summed over
// the steps; one column half after the other (16 accumulators and 16 link values live at a time).
// ONLY_OVER: only the steps whose log K_t exceeds safe_log_k (the matrix-core loop left exactly those out), added to
// what that loop found for the other steps (post[column half][v], the posterior sums of the lane's cells).
template <typename TL, bool ONLY_OVER>
__device__ __forceinline__ void grad_tile_direct(
    const float *al_f, const float *be_f, const double *ao, const double *bo, double Z, const TL *lk, TL *gl, float g,
    int L, int NBK, int Lb, int translen, int i0, int j0, int bi, int tlo, int thi, double safe, const float (*post)[16]) {
    const int lane = threadIdx.x, half = lane >> 5, l32 = lane & 31;
    const int bjA = (Lb - 1 - j0) / kBlk, bjB = bjA - 1;
    const int ia = i0 + l32 < Lb ? i0 + l32 : Lb - 1;
    const int pitch = translen - 1;
#pragma unroll 1
    for (int jh = 0; jh < 2; ++jh) {
        const int j = j0 + 32 * jh + l32, jb = j < Lb ? j : Lb - 1;
        const bool selA = (Lb - 1 - jb) / kBlk == bjA;
        const int dl = j - (i0 + 4 * half) - 1, pl = (i0 + 4 * half) * pitch + j - 1;
        auto valid = [&](int v) { return j < Lb && (unsigned)(dl - (8 * (v / 4) + (v % 4))) < (unsigned)translen; };
        auto index = [&](int v) { return pl + (8 * (v / 4) + (v % 4)) * pitch; };
        float e2[16], acc[16];   // E * log2(e) (-inf where there is no transition), sums
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            e2[v] = valid(v) ? to_float(lk[index(v)]) * kLog2e : DAGX_NEG_INF;
            acc[v] = ONLY_OVER ? post[jh][v] : 0.f;
        }
        // one step, given its block offsets (wave-uniform: ca = alpha block offset - Z; the two beta blocks' offsets) and
        // the step's residuals of this lane's column (rb) and row l32 (arow)
        auto one_step = [&](const double ca, const double cbA, const double cbB, const float rb, const float arow) __attribute__((always_inline)) {
            // beta side of the lane's column: residual + block offset + (alpha block offset - Z); -inf when dead
            const double kb = selA ? cbA : cbB;
            const double w = kb > (double)DAGX_NEG_INF ? (double)rb + (kb + ca) : (double)DAGX_NEG_INF;
            const int arow_bits = __builtin_bit_cast(int, arow);   // lane l32 (both halves) holds the residual of row i0 + l32
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = 8 * (v / 4) + (v % 4);                       // + 4 * half
                // (two reads of a fixed lane and a select: a cross-lane permute would make every one of the sixteen
                //  wait for its own round trip through the LDS crossbar)
                const float a_lo = __builtin_bit_cast(float, __builtin_amdgcn_readlane(arow_bits, row));
                const float a_hi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(arow_bits, row + 4));
                const double ad = (double)(half ? a_hi : a_lo);
                acc[v] += fast_exp2(__builtin_fmaf((float)(w + ad), kLog2e, e2[v]));
            }
        };
        if constexpr (!ONLY_OVER) {
            for (int t = tlo; t <= thi; ++t) {
                const double ca = ao[t * NBK + bi] - Z;
                const double cbA = bo[(t + 1) * NBK + bjA];
                const double cbB = bjB >= 0 ? bo[(t + 1) * NBK + bjB] : (double)DAGX_NEG_INF;
                if (!(ca > (double)DAGX_NEG_INF) || !(fmax(cbA, cbB) > (double)DAGX_NEG_INF)) continue;   // wave-uniform
                one_step(ca, cbA, cbB, be_f[t * L + jb], al_f[t * L + ia]);
            }
        } else {
            auto uniform_of = [&](const double x, const int src) -> double {   // lane src's value, in scalar registers
                const long long bits = __builtin_bit_cast(long long, x);
                const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(bits & 0xffffffffLL), src);
                const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(bits >> 32), src);
                return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)lo);
            };
            for (int g0 = tlo; g0 <= thi; g0 += kWave) {   // lane <-> step: which of these 64 steps were left out (as in step_scales)
                const bool live = g0 + lane <= thi;
                const int tl = live ? g0 + lane : thi;
                const double ca_l = ao[tl * NBK + bi] - Z, cbA_l = bo[(tl + 1) * NBK + bjA];
                const double cbB_l = bjB >= 0 ? bo[(tl + 1) * NBK + bjB] : (double)DAGX_NEG_INF;
                const double cbm = fmax(cbA_l, cbB_l);
                const bool dead = !live || !(ca_l > (double)DAGX_NEG_INF) || !(cbm > (double)DAGX_NEG_INF);
                unsigned long long over = __builtin_amdgcn_ballot_w64(!dead && !(ca_l + cbm <= safe));
                if (!over) continue;
                // the residual rows of a step are requested while the step before it is summed
                int k = __builtin_ctzll(over);
                float rb_n = be_f[(g0 + k) * L + jb], arow_n = al_f[(g0 + k) * L + ia];
                while (over) {
                    const int kc = k;
                    const float rb = rb_n, arow = arow_n;
                    over &= over - 1;
                    if (over) {
                        k = __builtin_ctzll(over);
                        rb_n = be_f[(g0 + k) * L + jb]; arow_n = al_f[(g0 + k) * L + ia];
                    }
                    one_step(uniform_of(ca_l, kc), uniform_of(cbA_l, kc), uniform_of(cbB_l, kc), rb, arow);
                }
            }
        }
#pragma unroll
        for (int v = 0; v < 16; ++v)
            if (valid(v)) gl[index(v)] = from_float<TL>(g * acc[v]);
    }
}

template <typename TL>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(5, 5)))
void dag_grad_links_tiles_kernel(GradTileArgs a) {
    // (the streaming workgroups come last in the grid: dispatched first they delay the tiles, 44 us against 39)
    if ((int)blockIdx.x >= a.tile_blocks) { grad_side_jobs(a, (int)blockIdx.x - a.tile_blocks); return; }
    const int tile_id = (int)blockIdx.x;
    // Workgroup id -> (sample, tile half) with the sample varying fastest: consecutive ids go to different
    // XCDs, so every XCD gets whole samples (balanced work, and a sample's tables stay in one L2).
    const int b = tile_id % a.B, q = tile_id / a.B;
    const int ih = q & 1, tidx = q >> 1;
    const int bi = a.tile_bi[tidx], jt = a.tile_jt[tidx];
    const int lane = threadIdx.x;
    const int L = a.L, T = a.T, translen = a.translen, NBK = a.NBK;
    const int Lb = (int)a.out_len[b], Tb = (int)a.tgt_len[b];
    const double Z = a.logz[a.B + b];
    if (!lengths_ok(Lb, Tb, L, T) || Tb < 2 || !finite_d(Z)) return;
    const int i0 = bi * kBlk + 32 * ih, j0 = jt * kBlk;
    // no (i < j < L_b, j - i <= translen) in this tile
    if (i0 >= Lb - 1 || j0 >= Lb || j0 + kBlk - 1 <= i0 || j0 - (i0 + 31) > translen) return;
    // operand layout of the 32x32x2 MFMA: lanes 0..31 carry step t, lanes 32..63 step t+1
    const int half = lane >> 5, l32 = lane & 31;
    // beta blocks of this tile's columns: positions L_b-1-j run downwards, at most two blocks
    const int bjA = (Lb - 1 - j0) / kBlk;
    const int bjB = bjA - 1;
    // Rows >= L_b and columns >= L_b are read through clamped (in-bounds) indices and not masked:
    // whatever they contribute lands in accumulator rows / columns that the epilogue never writes out.
    const int ia = i0 + l32 < Lb ? i0 + l32 : Lb - 1;
    const int jb0 = j0 + l32 < Lb ? j0 + l32 : Lb - 1, jb1 = j0 + 32 + l32 < Lb ? j0 + 32 + l32 : Lb - 1;
    const bool selA0 = (Lb - 1 - jb0) / kBlk == bjA, selA1 = (Lb - 1 - jb1) / kBlk == bjA;
    const char *al = reinterpret_cast<const char *>(a.ahat + (int64_t)b * T * L);
    const char *be = reinterpret_cast<const char *>(a.bhat + (int64_t)b * T * L + L);   // beta of step t+1
    const double *ao = a.aoff + (int64_t)b * T * NBK, *bo = a.boff + (int64_t)b * T * NBK;
    // The tile's link values are needed only after the step loop.  Those of the first column half are
    // fetched now, straight into LDS (no registers held across the loop), so that this read overlaps
    // the loop; the second half is loaded while the first is being finished.  Element (i, j) of the
    // sample sits at index i * (translen - 1) + j - 1; invalid cells read element 0.
    //   value v of column half jh: row i0 + 8 (v / 4) + 4 half + v % 4, column j0 + 32 jh + l32
    __shared__ unsigned landing[16 * kWave];
    const TL *lk = static_cast<const TL *>(a.links) + (int64_t)b * L * translen;
    const unsigned landing_lds = (unsigned)reinterpret_cast<uintptr_t>(landing);
    const int pitch = translen - 1;
    int dl[2], pl[2];   // per lane and column half: d and element index of the lane's first row
    bool jok[2];
#pragma unroll
    for (int jh = 0; jh < 2; ++jh) {
        const int j = j0 + 32 * jh + l32;
        jok[jh] = j < Lb;
        dl[jh] = j - (i0 + 4 * half) - 1;
        pl[jh] = (i0 + 4 * half) * pitch + j - 1;
    }
    auto cell_valid = [&](int jh, int v) { return jok[jh] && (unsigned)(dl[jh] - (8 * (v / 4) + (v % 4))) < (unsigned)translen; };
    auto cell_index = [&](int jh, int v) { return pl[jh] + (8 * (v / 4) + (v % 4)) * pitch; };
#pragma unroll
    for (int v = 0; v < 16; ++v)
        dma_elem<TL>(landing_lds + (unsigned)v * (kWave * 4u), lk, cell_valid(0, v) ? (unsigned)cell_index(0, v) * (unsigned)sizeof(TL) : 0u);
    f32x16 c0, c1;   // column halves
#pragma unroll
    for (int r = 0; r < 16; ++r) { c0[r] = 0.f; c1[r] = 0.f; }
    const int slack = Lb - Tb;
    // alpha[t][i] is alive for i - slack <= t <= i; beta[t+1][j] for j - slack - 1 <= t <= j - 1
    int tlo = j0 - slack - 1; if (tlo < i0 - slack) tlo = i0 - slack; if (tlo < 0) tlo = 0;
    int thi = i0 + 31; if (thi > Tb - 2) thi = Tb - 2;
    // Scale factors of kGroup steps at a time, worked out with lane <-> step (float64 arithmetic once
    // per step) and kept in LDS in log2 units:
    //   [0]: on exp(alpha_hat);  [1] / [2]: on exp(beta_hat) for the two beta blocks of the columns.
    // Steps past thi get -inf everywhere: both factors become 0, whatever row was loaded for them.
    constexpr int kGroup = kWave;
    __shared__ float scales[3][kGroup];
    const double safe = safe_log_k(thi - tlo + 1);   // log K_t up to which a step goes through the matrix product
    bool unsafe = false;   // wave-uniform: some step of the tile has log K_t > safe; those steps are left out of the loop
    auto step_scales = [&](int t0) {
        const int sl = lane;
        const bool live = t0 + sl <= thi;
        const int t = live ? t0 + sl : thi;
        const double ca = ao[t * NBK + bi], cbA = bo[(t + 1) * NBK + bjA];
        const double cbB = bjB >= 0 ? bo[(t + 1) * NBK + bjB] : (double)DAGX_NEG_INF;
        const double cbm = fmax(cbA, cbB);
        bool dead = !live || !(ca > (double)DAGX_NEG_INF) || !(cbm > (double)DAGX_NEG_INF);
        const bool over = !dead && !((ca - Z) + cbm <= safe);   // (the same expression as in grad_tile_direct; a NaN counts)
        unsafe = unsafe || __builtin_amdgcn_ballot_w64(over) != 0;
        dead = dead || over;
        const double xm = dead ? 0.0 : (ca - Z) + cbm;
        double h = 0.5 * xm; if (h > 64.0) h = 64.0;
        __syncthreads();   // the previous group's reads are done
        {
            scales[0][sl] = dead ? DAGX_NEG_INF : (float)h * kLog2e;
            scales[1][sl] = !dead && cbA > (double)DAGX_NEG_INF ? (float)((cbA - cbm) + (xm - h)) * kLog2e : DAGX_NEG_INF;
            scales[2][sl] = !dead && cbB > (double)DAGX_NEG_INF ? (float)((cbB - cbm) + (xm - h)) * kLog2e : DAGX_NEG_INF;
        }
        __syncthreads();
    };
    const float *fa_p = &scales[0][half], *fb0_p = &scales[selA0 ? 1 : 2][half], *fb1_p = &scales[selA1 ? 1 : 2][half];
    // Step pairs are loaded kDepth pairs before they are used (with several waves sharing a SIMD that
    // is a few microseconds, enough for a miss): the address is a wave-uniform row
    // offset plus a per-lane constant.  All loads are unconditional and in bounds: a pair whose second
    // step is past thi reads the row of its first step twice (beta) or the row after thi (alpha, which
    // exists: thi + 1 <= T_b - 1), and pairs wholly past the end repeat the last one.
    constexpr int kDepth = 8;
    const unsigned va = (unsigned)(half * L + ia) * 4u;
    const unsigned vb0 = (unsigned)(half * L + jb0) * 4u, vb1 = (unsigned)(half * L + jb1) * 4u;
    const unsigned vb0_single = (unsigned)jb0 * 4u, vb1_single = (unsigned)jb1 * 4u;
    float ra[kDepth], rb0[kDepth], rb1[kDepth];
    auto issue = [&](int k, int t) {   // t: first step of the pair
        const int tb = t < thi ? t : thi;
        const bool full = tb < thi;
        const unsigned row = (unsigned)(tb * L) * 4u;   // wave-uniform
        ra[k] = *reinterpret_cast<const float *>(al + row + va);
        rb0[k] = *reinterpret_cast<const float *>(be + row + (full ? vb0 : vb0_single));
        rb1[k] = *reinterpret_cast<const float *>(be + row + (full ? vb1 : vb1_single));
    };
    auto consume = [&](int k, int idx) {   // idx: index of the pair's first step in its group
        const float ea = fast_exp2(__builtin_fmaf(ra[k], kLog2e, fa_p[idx]));
        const float eb0 = fast_exp2(__builtin_fmaf(rb0[k], kLog2e, fb0_p[idx]));
        const float eb1 = fast_exp2(__builtin_fmaf(rb1[k], kLog2e, fb1_p[idx]));
        c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(ea, eb0, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(ea, eb1, c1, 0, 0, 0);
    };
    if (tlo <= thi) {
#pragma unroll
        for (int k = 0; k < kDepth; ++k) issue(k, tlo + 2 * k);
        for (int g0 = tlo; g0 <= thi; g0 += kGroup) {
            step_scales(g0);
            // (the inner loop holds no loads but the ring's, so that the compiler can count them)
            const int gend = g0 + kGroup - 1 < thi ? g0 + kGroup - 1 : thi;
            for (int t = g0; t <= gend; t += 2 * kDepth) {
                const int idx0 = t - g0;                    // multiple of 16
#pragma unroll
                for (int k = 0; k < kDepth; ++k) {
                    consume(k, idx0 + 2 * k);               // pairs wholly past the end add zeros
                    issue(k, t + 2 * k + 2 * kDepth);
                    __builtin_amdgcn_sched_barrier(0);      // keep each refill where it is: kDepth - 1 pairs ahead of its use
                }
            }
        }
    }
    // epilogue: multiply by P = exp(E) and the upstream gradient, write the valid part of the tile
    const float g = a.grad_out[b * a.gstride];
    TL *gl = static_cast<TL *>(a.grad_links) + (int64_t)b * L * translen;
    wait_vmem_all();     // the link values of the first column half have landed
    __syncthreads();
    TL second[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) second[v] = lk[cell_valid(1, v) ? cell_index(1, v) : 0];
    auto link_of = [&](int jh, int v) -> float { return jh ? to_float(second[v]) : dma_decode<TL>(landing[v * kWave + lane]); };
    bool overflowed;
    {   // a sum that is not a finite number in a cell this wave writes: the bound rules that out for finite tables
        bool bad = false;
#pragma unroll
        for (int v = 0; v < 16; ++v)
            bad = bad || (cell_valid(0, v) && !(c0[v] <= 3.0e38f)) || (cell_valid(1, v) && !(c1[v] <= 3.0e38f));
        overflowed = __builtin_amdgcn_ballot_w64(bad) != 0;
    }
    if (__builtin_expect(overflowed, 0)) {   // a NaN in the tables: the whole tile, every step in the direct form
        grad_tile_direct<TL, false>(reinterpret_cast<const float *>(al), reinterpret_cast<const float *>(be), ao, bo, Z, lk, gl, g,
                                    L, NBK, Lb, translen, i0, j0, bi, tlo, thi, safe, nullptr);
        return;
    }
    // posterior sums of the lane's cells of one column half: the loop's sums times P = exp(E)
    auto posteriors = [&](auto all_valid, int jh, const f32x16 &c, float (&post)[16]) __attribute__((always_inline)) {
        // transitions too small for exp() in float32 take their factor through the logarithm of the sum
        bool tiny = false;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float e = link_of(jh, v);
            tiny = tiny || ((decltype(all_valid)::value || cell_valid(jh, v)) && e < -80.f && e > DAGX_NEG_INF);
        }
        const bool any_tiny = __builtin_amdgcn_ballot_w64(tiny) != 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const bool valid = decltype(all_valid)::value || cell_valid(jh, v);
            const float e = link_of(jh, v);
            post[v] = valid ? c[v] * fast_exp2(e * kLog2e) : 0.f;
            if (any_tiny && valid && e < -80.f) post[v] = (c[v] > 0.f && e > DAGX_NEG_INF) ? fast_exp2(__builtin_fmaf(e, kLog2e, fast_log2(c[v]))) : 0.f;
        }
    };
    if (__builtin_expect(unsafe, 0)) {   // the steps the loop left out, in the direct form, on top of the loop's sums
        float post[2][16];
        posteriors(std::false_type{}, 0, c0, post[0]);
        posteriors(std::false_type{}, 1, c1, post[1]);
        grad_tile_direct<TL, true>(reinterpret_cast<const float *>(al), reinterpret_cast<const float *>(be), ao, bo, Z, lk, gl, g,
                                   L, NBK, Lb, translen, i0, j0, bi, tlo, thi, safe, post);
        return;
    }
    auto finish = [&](auto all_valid, int jh, const f32x16 &c) {
        float post[16];
        posteriors(all_valid, jh, c, post);
#pragma unroll
        for (int v = 0; v < 16; ++v)
            if (decltype(all_valid)::value || cell_valid(jh, v)) gl[cell_index(jh, v)] = from_float<TL>(g * post[v]);
    };
#pragma unroll
    for (int jh = 0; jh < 2; ++jh) {
        const int jlo = j0 + 32 * jh;
        // every cell of the 32x32 block valid (wave-uniform): no per-element predicates
        const bool interior = jlo + 31 < Lb && jlo - (i0 + 31) - 1 >= 0 && jlo + 31 - i0 - 1 < translen;
        if (interior) finish(std::true_type{}, jh, jh ? c1 : c0);
        else finish(std::false_type{}, jh, jh ? c1 : c0);
    }
}


// ---- host side ------------------------------------------------------------------------------
static int check_common(const void *match, int mdt, const int64_t *ms, const void *links, int ldt,
                        const int64_t *ol, const int64_t *tl, int B, int T, int L, int translen, const char *who) {
    if (B < 0 || T < 1 || L < 1 || translen < 1) { set_error("%s: bad sizes B=%d T=%d L=%d translen=%d", who, B, T, L, translen); return DAGX_ERR_ARGUMENT; }
    if (B > 0 && (!match || !ms || !links || !ol || !tl)) { set_error("%s: null pointer argument", who); return DAGX_ERR_ARGUMENT; }
    if (mdt < DAGX_F32 || mdt > DAGX_BF16 || ldt < DAGX_F32 || ldt > DAGX_BF16) { set_error("%s: unsupported dtype", who); return DAGX_ERR_ARGUMENT; }
    if (L > 8192) { set_error("%s: graph size L=%d exceeds the supported 8192", who, L); return DAGX_ERR_UNSUPPORTED; }
    if (B > 65535 || T > 65535) { set_error("%s: B and T must not exceed 65535", who); return DAGX_ERR_UNSUPPORTED; }
    return DAGX_OK;
}


static bool force_exact() { return force_log_domain(); }

// ticket + launch counter (16 ints), 2*B*C progress words, B "left" counters, B risk words; rounded to 8 bytes
static size_t sweep_sync_ints(int B, int C) { return ((16 + (size_t)2 * B * C + (size_t)2 * B) + 1) & ~(size_t)1; }

// ticket + progress words (rounded to 8 bytes), then the fast kernel's two read-outs per sample
static size_t sweep_bytes(int B, int C) { return sweep_sync_ints(B, C) * sizeof(int) + (size_t)2 * B * sizeof(double); }

// For table 0.  Tables with more groups are used where the caller's workspace has room for them: a buffer that is large enough for the
// largest graph must stay large enough for smaller ones, whose tables may have more groups.
size_t loss_fwd_workspace_bytes(int B, int T, int L, int translen) {
    (void)T;
    const int C = sweep_groups(B, L, translen);
    return C > 0 ? sweep_bytes(B, C) : 0;
}
static int groups_that_fit(int B, size_t workspace_bytes) {
    int C = kMaxGroups;
    while (C > 0 && sweep_bytes(B, C) > workspace_bytes) --C;
    return C;
}

size_t loss_bwd_workspace_bytes(int B) { (void)B; return 0; }

// The tile kernel's dynamic LDS (transpose patches while the tiles are staged, step buffers afterwards) exceeds the
// default limit: the limit is raised once per device and instantiation (not a call a graph capture may contain;
// dagx_prepare_device does it for every instantiation ahead of time).
template <typename TM, typename TL, bool WIDE>
static int prepare_tiles_kernel() {
    static std::atomic<unsigned long long> attr_set{0};   // per template instantiation: one bit per device
    int device = 0;
    (void)hipGetDevice(&device);
    const unsigned long long bit = 1ull << (device & 63);
    if (!(attr_set.load(std::memory_order_acquire) & bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(dag_sweep_tiles_kernel<TM, TL, WIDE>), hipFuncAttributeMaxDynamicSharedMemorySize, kChunkLdsBytes);
        if (e != hipSuccess) { set_error("dag_loss_fwd: cannot reserve %d bytes of LDS: %s", kChunkLdsBytes, hipGetErrorString(e)); return DAGX_ERR_LAUNCH; }
        attr_set.fetch_or(bit, std::memory_order_release);
    }
    return DAGX_OK;
}
template <typename TM>
static int prepare_tiles_kernels_of() {
    int rc = prepare_tiles_kernel<TM, float, false>();
    if (!rc) rc = prepare_tiles_kernel<TM, __half, false>();
    if (!rc) rc = prepare_tiles_kernel<TM, bf16_t, false>();
    if (!rc) rc = prepare_tiles_kernel<TM, float, true>();
    if (!rc) rc = prepare_tiles_kernel<TM, __half, true>();
    if (!rc) rc = prepare_tiles_kernel<TM, bf16_t, true>();
    return rc;
}

template <typename TM, typename TL>
static int launch_sweeps(SweepArgs base, size_t workspace_bytes, hipStream_t st) {
    TileSweepArgs a{};
    static_cast<SweepArgs &>(a) = base;
    int C = force_exact() ? 0 : sweep_groups(a.B, a.L, a.translen);
    // the tile kernel indexes match with 32-bit arithmetic
    const int64_t span = (int64_t)(a.T - 1) * (a.ms1 < 0 ? -a.ms1 : a.ms1) + (int64_t)(a.L - 1) * (a.ms2 < 0 ? -a.ms2 : a.ms2);
    if (span >= (1LL << 31) / (int64_t)sizeof(TM) || a.ms1 < 0 || a.ms2 < 0) C = 0;
    if ((int64_t)a.B * a.L * a.translen < 4) C = 0;   // (the tiles are loaded four elements at a time)
    int rc;
    if (C == 0) {   // every sample goes to the log-domain kernel
        hipLaunchKernelGGL(dag_fill_int_kernel, dim3((a.B + 255) / 256), dim3(256), 0, st, a.flags, a.B, 1);
        if ((rc = check_launch("dag_fill"))) return rc;
    }
    if (C > 0) {
        // Two sweeps per sample whose read-outs bracket log Z.  With gradients they are the alpha sweep (rounding
        // up) and the beta sweep (rounding down; its read-out is the loss, as in fs_plugins/custom_ops/dag_loss.py:106-109).
        // Without, the reference runs the alpha sweep alone (dag_loss.cu:346-371); here a second alpha sweep that
        // rounds up rides along, so that the value returned is never one the linear domain has silently cut short.
        a.ndir = 2;
        a.rev[0] = 0; a.rev[1] = a.loss_dir ? 1 : 0;
        a.upper[0] = a.loss_dir ? 1 : 0; a.upper[1] = a.loss_dir ? 0 : 1;
        const int B8 = (a.B + 7) & ~7, room = groups_that_fit(a.B, workspace_bytes);
        auto plan_for = [&](const bool wide) {
            make_tables<1>(a.table, a.choice, a.B, a.T, a.L, a.translen, C, room, kSweepCosts, wide);
            a.C = a.choice.most;
            a.zfast = reinterpret_cast<double *>(a.sync + sweep_sync_ints(a.B, a.C));   // (zero again behind every launch, as the words in front)
        };
        plan_for(float64_first());
        if ((rc = prepare_tiles_kernel<TM, TL, false>()) || (rc = prepare_tiles_kernel<TM, TL, true>())) return rc;
        if (!float64_first()) {
            a.only_flagged = 0;
            hipLaunchKernelGGL((dag_sweep_tiles_kernel<TM, TL, false>), dim3(a.ndir * B8 * a.C), dim3(kTileWaves * kWave), kChunkLdsBytes, st, a);
            if ((rc = check_launch("dag_sweep_tiles"))) return rc;
        } else {   // the caller knows its inputs for sharply peaked: no float32 pass whose result would not stand
            hipLaunchKernelGGL(dag_mark_all_kernel, dim3((a.B + 255) / 256), dim3(256), 0, st, a.flags, a.B, a.sync);
            if ((rc = check_launch("dag_mark_all"))) return rc;
        }
        // the samples whose two read-outs did not agree, once more with float64 linear-domain numbers (the pipeline
        // words are zero again, as the first launch found them)
        a.only_flagged = 1;
        if (!float64_first()) plan_for(true);
        hipLaunchKernelGGL((dag_sweep_tiles_kernel<TM, TL, true>), dim3(a.ndir * B8 * a.C), dim3(kTileWaves * kWave), kChunkLdsBytes, st, a);
        if ((rc = check_launch("dag_sweep_tiles (wide)"))) return rc;
    }
    constexpr int NT = 1024;
    base = a;
    base.only_flagged = 1;
    const size_t lds = (size_t)a.L * 2 * sizeof(double);
    auto exact_kernel = dag_sweep_exact_kernel<TM, TL, NT>;
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(exact_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) { set_error("dag_loss_fwd: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e)); return DAGX_ERR_LAUNCH; }
    }
    hipLaunchKernelGGL(exact_kernel, dim3(a.B, a.loss_dir ? 2 : 1), dim3(NT), lds, st, base);
    return check_launch("dag_sweep_exact");
}

template <typename TM>
static int dispatch_links(int ldt, const SweepArgs &a, size_t workspace_bytes, hipStream_t st) {
    switch (ldt) {
        case DAGX_F32: return launch_sweeps<TM, float>(a, workspace_bytes, st);
        case DAGX_F16: return launch_sweeps<TM, __half>(a, workspace_bytes, st);
        default: return launch_sweeps<TM, bf16_t>(a, workspace_bytes, st);
    }
}

struct BwdArgs {
    const float *go; int64_t gs;
    const float *ahat, *bhat; const double *aoff, *boff, *logz;
    const int64_t *ol, *tl; int B, T, L, translen, NBK;
};

static bool grad_tiles_apply(int L) { return !force_exact() && (L + kBlk - 1) / kBlk <= kMaxBlocksFast; }

// what has to be cleared in front of the grad_links tile kernel
static ZeroJob make_zero_job(const BwdArgs &g, void *gl, size_t elem) {
    int chunks = g.L < 32 ? g.L : 32;
    const int rows = (g.L + chunks - 1) / chunks;
    chunks = (g.L + rows - 1) / rows;
    return ZeroJob{static_cast<unsigned char *>(gl), (int)elem, g.ol, g.tl, g.logz, g.B, g.T, g.L, g.translen,
                   rows, chunks, g.B * chunks};
}

template <typename TM>
static int launch_grad_match(const BwdArgs &g, const void *match, const int64_t *ms, void *gm, const ZeroJob &zero, hipStream_t st) {
    const int64_t blocks = (int64_t)zero.blocks + (int64_t)((g.L + 255) / 256) * g.T * g.B;
    if (blocks > 0x7fffffffLL) { set_error("dag_loss_bwd: B*T*L too large for one launch"); return DAGX_ERR_UNSUPPORTED; }
    hipLaunchKernelGGL((dag_grad_match_kernel<TM>), dim3((unsigned)blocks), dim3(256), 0, st, g.go, g.gs,
                       g.ahat, g.bhat, g.aoff, g.boff, g.logz, static_cast<const TM *>(match), ms[0], ms[1], ms[2],
                       g.ol, g.tl, g.B, g.T, g.L, g.NBK, static_cast<TM *>(gm), zero);
    return check_launch("dag_grad_match");
}

// match / ms / match_dtype / gm: grad_match to be computed in the same launch as the tiles (gm == nullptr: not asked for,
// or already done by a launch of its own)
template <typename TL>
static int launch_grad_links(const BwdArgs &g, const void *links, void *gl, const void *match, const int64_t *ms,
                             int match_dtype, void *gm, hipStream_t st) {
    if (grad_tiles_apply(g.L)) {
        // block-scaled tiles (with their own direct-form redo); zeros where no tile writes and grad_match from
        // workgroups of the same launch
        GradTileArgs ta{g.go, g.gs, g.ahat, g.bhat, g.aoff, g.boff, g.logz, links, gl, g.ol, g.tl,
                        g.B, g.T, g.L, g.translen, g.NBK};
        ta.zero = make_zero_job(g, gl, sizeof(TL));
        ta.match = match; ta.match_dtype = match_dtype; ta.grad_match = gm;
        if (gm) { ta.ms0 = ms[0]; ta.ms1 = ms[1]; ta.ms2 = ms[2]; }
        const int NB = (g.L + kBlk - 1) / kBlk;
        int W = (g.translen + kBlk - 1) / kBlk; if (W > NB - 1) W = NB - 1;
        ta.ntile = 0;
        for (int bi = 0; bi < NB; ++bi)
            for (int jt = bi; jt <= bi + W && jt < NB; ++jt) { ta.tile_bi[ta.ntile] = (unsigned char)bi; ta.tile_jt[ta.ntile] = (unsigned char)jt; ++ta.ntile; }
        ta.tile_blocks = 2 * ta.ntile * g.B;   // two row halves per tile
        const int64_t match_blocks = gm ? (int64_t)((g.L + 255) / 256) * g.T * g.B : 0;
        const int64_t blocks = (int64_t)ta.tile_blocks + ta.zero.blocks + match_blocks;
        if (blocks > 0x7fffffffLL) { set_error("dag_loss_bwd: B*T*L too large for one launch"); return DAGX_ERR_UNSUPPORTED; }
        ta.match_blocks = (int)match_blocks;
        hipLaunchKernelGGL((dag_grad_links_tiles_kernel<TL>), dim3((unsigned)blocks), dim3(kWave), 0, st, ta);
        return check_launch("dag_grad_links_tiles");
    }
    // direct (log-domain) form: graphs beyond the tile kernels, or the log-domain-only mode
    constexpr int RI = 32;
    hipLaunchKernelGGL((dag_grad_links_kernel<TL, RI>), dim3((g.translen + 63) / 64, (g.L + RI - 1) / RI, g.B), dim3(256), 0, st,
                       g.go, g.gs, g.ahat, g.bhat, g.aoff, g.boff, g.logz, static_cast<const TL *>(links), g.ol, g.tl,
                       g.B, g.T, g.L, g.translen, g.NBK, static_cast<TL *>(gl));
    return check_launch("dag_grad_links");
}

}  // namespace dagx

using namespace dagx;


static int loss_fwd_impl(const void *match, int match_dtype, const int64_t match_strides[3],
                         const void *links, int links_dtype,
                         const int64_t *out_len, const int64_t *tgt_len,
                         int B, int T, int L, int translen,
                         float *alpha_hat, float *beta_hat, double *alpha_off, double *beta_off,
                         double *logz, float *loss, int *sample_flags, int require_gradient,
                         void *workspace, size_t workspace_bytes, void *stream) {
    int rc = check_common(match, match_dtype, match_strides, links, links_dtype, out_len, tgt_len, B, T, L, translen, "dag_loss_fwd");
    if (rc) return rc;
    if (B == 0) return DAGX_OK;                 // an empty batch owns no memory: nothing to check or launch
    if (!alpha_hat || !beta_hat || !alpha_off || !beta_off || !logz || !loss || !sample_flags) { set_error("dag_loss_fwd: an output pointer is null"); return DAGX_ERR_ARGUMENT; }
    size_t need = loss_fwd_workspace_bytes(B, T, L, translen);
    if (need > 0 && (!workspace || workspace_bytes < need)) { set_error("dag_loss_fwd: workspace of %zu bytes required, %zu given", need, workspace_bytes); return DAGX_ERR_WORKSPACE; }
    SweepArgs a{};
    a.match = match; a.ms0 = match_strides[0]; a.ms1 = match_strides[1]; a.ms2 = match_strides[2];
    a.links = links; a.out_len = out_len; a.tgt_len = tgt_len;
    a.B = B; a.T = T; a.L = L; a.translen = translen; a.NBK = (L + kBlk - 1) / kBlk;
    a.hat[0] = alpha_hat; a.hat[1] = beta_hat; a.off[0] = alpha_off; a.off[1] = beta_off;
    a.logz = logz; a.loss = loss; a.loss_dir = require_gradient ? 1 : 0; a.flags = sample_flags; a.sync = static_cast<int *>(workspace);
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (match_dtype) {
        case DAGX_F32: return dispatch_links<float>(links_dtype, a, workspace_bytes, st);
        case DAGX_F16: return dispatch_links<__half>(links_dtype, a, workspace_bytes, st);
        default: return dispatch_links<bf16_t>(links_dtype, a, workspace_bytes, st);
    }
}

extern "C" int dagx_loss_fwd(const void *match, int match_dtype, const int64_t match_strides[3],
                             const void *links, int links_dtype,
                             const int64_t *out_len, const int64_t *tgt_len,
                             int B, int T, int L, int translen,
                             float *alpha_hat, float *beta_hat, double *alpha_off, double *beta_off,
                             double *logz, float *loss, int *sample_flags, int require_gradient,
                             void *workspace, size_t workspace_bytes, void *stream) {
    return loss_fwd_impl(match, match_dtype, match_strides, links, links_dtype, out_len, tgt_len, B, T, L, translen,
                         alpha_hat, beta_hat, alpha_off, beta_off, logz, loss, sample_flags, require_gradient,
                         workspace, workspace_bytes, stream);
}

// ---- the forward for callers that cannot allocate ------------------------------------------------------
// The pipeline words and read-outs of the tile sweeps (what dagx_loss_fwd takes as `workspace`) in a
// device array owned by the library: every GPU the library runs on holds its own copy until the process
// ends.  Zero when the code object is loaded; the sweep kernel leaves every word it used zero again.
constexpr size_t kScratchBytes = 128 * 1024;
// (What fits is decided as for groups of any number of blocks; groups of at most eight can be one more, 40 bytes a sample
//  instead of 32.)
constexpr size_t kScratchHeld = kScratchBytes / 4 * 5 + 256;
static __device__ __align__(256) unsigned char scratch[kScratchHeld];

constexpr int kMaxDevices = 64;
static std::atomic<void *> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (looked up once per device; in host code the
// array's name is only a handle for this lookup, never an address a kernel may be given).
static int scratch_of_current_device(void **out) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) { set_error("dag_loss_fwd_noalloc: hipGetDevice failed: %s", hipGetErrorString(e)); return DAGX_ERR_LAUNCH; }
    if (device < 0 || device >= kMaxDevices) { set_error("dag_loss_fwd_noalloc: device index %d not supported (max %d)", device, kMaxDevices - 1); return DAGX_ERR_UNSUPPORTED; }
    void *p = g_scratch_ptr[device].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) { set_error("dag_loss_fwd_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e)); return DAGX_ERR_LAUNCH; }
        g_scratch_ptr[device].store(p, std::memory_order_release);   // a concurrent first call stores the same address
    }
    *out = p;
    return DAGX_OK;
}

extern "C" size_t dagx_loss_fwd_noalloc_max_bytes(void) { return kScratchBytes; }

// Everything the forward entry points do once per device, done now: the LDS limit of every instantiation of the tile
// kernel and the address of the built-in scratch array.  After it, dagx_loss_fwd / dagx_loss_fwd_noalloc on this
// device make kernel launches only (for L <= 3072), which is what a stream capture may hold.
extern "C" int dagx_prepare_device(void) {
    int rc = prepare_tiles_kernels_of<float>();
    if (!rc) rc = prepare_tiles_kernels_of<__half>();
    if (!rc) rc = prepare_tiles_kernels_of<bf16_t>();
    if (!rc) rc = prepare_align_kernels();
    void *ptr = nullptr;
    if (!rc) rc = scratch_of_current_device(&ptr);
    return rc;
}

// Zero-fill of a workspace for dagx_loss_fwd (a kernel launch on `stream`; needed once per buffer, before its first use).
extern "C" int dagx_loss_fwd_init_workspace(void *workspace, size_t workspace_bytes, void *stream) {
    if (workspace_bytes == 0) return DAGX_OK;
    if (!workspace || (workspace_bytes & 3) || (reinterpret_cast<uintptr_t>(workspace) & 7)) { set_error("dag_loss_fwd_init_workspace: needs an 8-byte aligned buffer of a multiple of 4 bytes"); return DAGX_ERR_ARGUMENT; }
    const size_t n = workspace_bytes / 4;
    if (n > 0x7fffffffu) { set_error("dag_loss_fwd_init_workspace: buffer too large"); return DAGX_ERR_ARGUMENT; }
    hipLaunchKernelGGL(dag_fill_int_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<int *>(workspace), (int)n, 0);
    return check_launch("dag_fill");
}

extern "C" int dagx_loss_fwd_noalloc(const void *match, int match_dtype, const int64_t match_strides[3],
                                     const void *links, int links_dtype,
                                     const int64_t *out_len, const int64_t *tgt_len,
                                     int B, int T, int L, int translen,
                                     float *alpha_hat, float *beta_hat, double *alpha_off, double *beta_off,
                                     double *logz, float *loss, int *sample_flags, int require_gradient,
                                     void *stream) {
    if (B < 0 || T < 1 || L < 1 || translen < 1) { set_error("dag_loss_fwd_noalloc: bad sizes B=%d T=%d L=%d translen=%d", B, T, L, translen); return DAGX_ERR_ARGUMENT; }
    const size_t need = loss_fwd_workspace_bytes(B, T, L, translen);
    const int C = groups_needed(L, translen, kMaxBlocksFast);
    const size_t asked = C > 0 ? sweep_bytes(B, C) : 0;
    if (asked > kScratchBytes || need > kScratchHeld) {
        set_error("dag_loss_fwd_noalloc: B=%d, L=%d needs %zu bytes of pipeline words, the built-in scratch holds %zu "
                  "(use dagx_loss_fwd with a caller workspace)", B, L, asked, kScratchBytes);
        return DAGX_ERR_UNSUPPORTED;
    }
    void *ptr = nullptr;
    if (need > 0) {
        const int rc = scratch_of_current_device(&ptr);
        if (rc) return rc;
    }
    return loss_fwd_impl(match, match_dtype, match_strides, links, links_dtype, out_len, tgt_len, B, T, L, translen,
                         alpha_hat, beta_hat, alpha_off, beta_off, logz, loss, sample_flags, require_gradient,
                         ptr, need > 0 ? kScratchHeld : 0, stream);
}

extern "C" int dagx_loss_bwd(const float *grad_out, int64_t grad_out_stride,
                             const float *alpha_hat, const float *beta_hat,
                             const double *alpha_off, const double *beta_off, const double *logz,
                             const int *sample_flags,
                             const void *match, int match_dtype, const int64_t match_strides[3],
                             const void *links, int links_dtype,
                             const int64_t *out_len, const int64_t *tgt_len,
                             int B, int T, int L, int translen,
                             void *grad_match, void *grad_links,
                             void *workspace, size_t workspace_bytes, void *stream) {
    int rc = check_common(match, match_dtype, match_strides, links, links_dtype, out_len, tgt_len, B, T, L, translen, "dag_loss_bwd");
    if (rc) return rc;
    if (B == 0) return DAGX_OK;
    if (!grad_out || !alpha_hat || !beta_hat || !alpha_off || !beta_off || !logz) { set_error("dag_loss_bwd: a saved-state pointer is null"); return DAGX_ERR_ARGUMENT; }
    (void)workspace; (void)workspace_bytes; (void)sample_flags;   // the backward needs no scratch
    hipStream_t st = static_cast<hipStream_t>(stream);
    BwdArgs g{grad_out, grad_out_stride, alpha_hat, beta_hat, alpha_off, beta_off, logz, out_len, tgt_len,
              B, T, L, translen, (L + kBlk - 1) / kBlk};
    // With both gradients asked for and the tile kernel in charge, grad_match rides in its launch.
    const bool together = grad_match && grad_links && grad_tiles_apply(L);
    if (grad_match && !together) {
        ZeroJob zero{};
        switch (match_dtype) {
            case DAGX_F32: rc = launch_grad_match<float>(g, match, match_strides, grad_match, zero, st); break;
            case DAGX_F16: rc = launch_grad_match<__half>(g, match, match_strides, grad_match, zero, st); break;
            default: rc = launch_grad_match<bf16_t>(g, match, match_strides, grad_match, zero, st); break;
        }
        if (rc) return rc;
    }
    if (grad_links) {
        switch (links_dtype) {
            case DAGX_F32: rc = launch_grad_links<float>(g, links, grad_links, match, match_strides, match_dtype, together ? grad_match : nullptr, st); break;
            case DAGX_F16: rc = launch_grad_links<__half>(g, links, grad_links, match, match_strides, match_dtype, together ? grad_match : nullptr, st); break;
            default: rc = launch_grad_links<bf16_t>(g, links, grad_links, match, match_strides, match_dtype, together ? grad_match : nullptr, st); break;
        }
    }
    return rc;
}
