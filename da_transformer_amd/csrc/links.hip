// Transition log-probabilities from per-head scores (the tail of the link predictor), gfx950.
//
//   links[b][i][d] = LSE_c( content[b][i][j][c] - LSE_{j' in win(b,i)} content[b][i][j'][c] + log_gates[b][i][c] ),
//   j = i + d + 1,  win(b,i) = { j : i < j < min(valid_end[b][i], i + 1 + translen, L) },  -inf outside the window.
//
// This is what fs_plugins/models/glat_decomposed_with_link.py:380-404 computes with a masked_fill, a
// gather into the shifted layout (:319-335), a log_softmax over the transitions, an add and a
// logsumexp over the heads -- each a pass over a [B,L,translen,H] float tensor.  Here a row (b, i) is
// read once: its window is H * n contiguous elements of `content`, held in registers by one, two or four
// waves (four window positions a lane, so that a row leaves room for enough other rows on a SIMD to cover its loads).
// HBM-bound once the waves in flight suffice: the forward reads the windows and writes [B,L,translen]; the backward reads
// the windows again and writes the gradient over the whole [B,L,L,H] tensor in place (zeros outside the windows), as the
// dense batched-GEMM backward that follows it expects.
// Measured, forward behind backward in the same storage, lengths between 3/4 L and L, against one wave per row with the
// whole window in registers (2 waves a SIMD), three exponentials per score in the backward and cached zeros: B=64 L=512
// H=8 float32 254 -> 218 us, B=32 118 -> 80, float16 B=64 215 -> 118; B=16 L=1024 H=8 float16 229 -> 98; B=8 L=512 H=16
// float32 76 -> 47.  Between the copy that lays the scores out and the one that takes the gradient, those included: 803 ->
// 780, 408 -> 381, 586 -> 475, 602 -> 474, 228 -> 203.  Non-temporal stores of the gradient inside the window were slower.
#include <type_traits>

#include "dagx_common.h"

namespace dagx {

constexpr int kLinkThreads = 256;                 // four waves, one row each
constexpr int kLinkWaves = kLinkThreads / kWave;

// ---- reductions of one value per head over the 64 lanes --------------------------------------------
// The heads are shared out while they are reduced: in every step a lane keeps half of its heads, hands the other half to
// its partner and takes the partner's half of its own (7 operations for 8 heads where reducing every head by itself takes 48).
// The partners are lane ^ 15, ^ 7, ^ 3, ^ 1 (DPP row_mirror, row_half_mirror, quad_perm): each differs from the lane in the
// step's bit and agrees in the ones before it.  Afterwards lane l holds the total of head head_of<H>(l).
template <int CTRL>
__device__ __forceinline__ float dpp_lane(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int H> __device__ __forceinline__ int head_of(int lane) { return (lane & 15) / (16 / H); }
template <int H> __device__ __forceinline__ constexpr int lane_of(int head) { return head * (16 / H); }
struct OpMax { static __device__ __forceinline__ float apply(float a, float b) { return fmaxf(a, b); } };
struct OpSum { static __device__ __forceinline__ float apply(float a, float b) { return a + b; } };
template <typename OP, int CTRL, int N>
__device__ __forceinline__ void share_step(float (&v)[N], bool upper) {   // v[0 .. N/2) <- the lane's half, with the partner's values
    if constexpr (N > 1) {
#pragma unroll
        for (int c = 0; c < N / 2; ++c) {
            const float mine = upper ? v[c + N / 2] : v[c], other = upper ? v[c] : v[c + N / 2];
            v[c] = OP::apply(mine, dpp_lane<CTRL>(other));
        }
    } else {
        v[0] = OP::apply(v[0], dpp_lane<CTRL>(v[0]));
    }
}
template <typename OP, int H>
__device__ __forceinline__ float lanes_share(const float (&v)[H], int lane) {
    float a[H], b[H > 2 ? H / 2 : 1], c[H > 4 ? H / 4 : 1], d[H > 8 ? H / 8 : 1];
#pragma unroll
    for (int k = 0; k < H; ++k) a[k] = v[k];
    share_step<OP, 0x140, H>(a, lane & 8);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(b) / 4); ++k) b[k] = a[k];
    share_step<OP, 0x141>(b, lane & 4);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(c) / 4); ++k) c[k] = b[k];
    share_step<OP, 0x1B>(c, lane & 2);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(d) / 4); ++k) d[k] = c[k];
    share_step<OP, 0xB1>(d, lane & 1);
    float t = d[0];
    t = OP::apply(t, __shfl_xor(t, 16, kWave));
    t = OP::apply(t, __shfl_xor(t, 32, kWave));
    return t;
}
// the value that the lanes of head c hold, wave-uniform
template <int H>
__device__ __forceinline__ void lanes_spread(float t, float (&v)[H]) {
#pragma unroll
    for (int c = 0; c < H; ++c) v[c] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, t), lane_of<H>(c)));
}

// The H scores of one window position, as floats (one or two 16-byte loads for the usual H).
template <typename TC, int H>
__device__ __forceinline__ void load_heads(const TC *p, float (&x)[H]) {
    struct alignas(sizeof(TC) * H >= 16 ? 16 : sizeof(TC) * H) Pack { TC v[H]; };
    const Pack raw = *reinterpret_cast<const Pack *>(p);
#pragma unroll
    for (int c = 0; c < H; ++c) x[c] = to_float(raw.v[c]);
}
template <typename TC, int H>
__device__ __forceinline__ void store_heads(TC *p, const float (&x)[H]) {
    struct alignas(sizeof(TC) * H >= 16 ? 16 : sizeof(TC) * H) Pack { TC v[H]; };
    Pack raw;
#pragma unroll
    for (int c = 0; c < H; ++c) raw.v[c] = from_float<TC>(x[c]);
    *reinterpret_cast<Pack *>(p) = raw;
}

struct LinkRow { int b, i, jlo, n; };
__device__ __forceinline__ LinkRow link_row(const int64_t *valid_end, int64_t row, int L, int translen) {
    LinkRow r;
    r.b = (int)(row / L); r.i = (int)(row % L);
    r.jlo = r.i + 1;
    int64_t e = valid_end[row];
    int jhi = e < (int64_t)L ? (int)(e < 0 ? 0 : e) : L;
    if (jhi > r.jlo + translen) jhi = r.jlo + translen;
    r.n = jhi > r.jlo ? jhi - r.jlo : 0;
    return r;
}

constexpr int kLinkPer = 4;                       // window positions per lane
// Sums of products of probabilities are taken as they are down to 2^-100 times the largest factor that a gate puts before a
// probability (1 at least): a probability that left the float32 range (below 2^-126) still does not count there, whatever
// its gate.  Below that, and above kLinkHuge, which gates of at most 0 never reach, a position takes the route through its
// largest term.
// kLinkMostGrad: 2^26; over a sum of at least 2^-100 times the largest factor, and times that factor, it is still finite.
constexpr float kLinkTiny = 7.8886091e-31f, kLinkHuge = 64.0f, kLinkMostGrad = 67108864.0f;
template <int H>
__device__ __forceinline__ float least_sum(float own, const float (&factor)[H]) {   // own: the factor of the lane's head
    float most = 1.0f;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(own > 1.0f) != 0, 0))
#pragma unroll
        for (int c = 0; c < H; ++c) most = fmaxf(most, factor[c]);
    return kLinkTiny * most;
}

// links and lse (the per-head log normalisers, [B][L][H], kept for the backward).  WPR waves share a row: wave `sub` has
// the chunks sub, sub + WPR, ... of 64 window positions; min(translen, L - 1) <= 64 * kLinkPer * WPR.
template <typename TC, int H, int WPR>
__global__ __launch_bounds__(kLinkThreads) void links_fwd_kernel(
    const TC *__restrict__ content, const float *__restrict__ log_gates, const int64_t *__restrict__ valid_end,
    int64_t rows, int L, int translen, TC *__restrict__ links, float *__restrict__ lse_out) {
    __shared__ float2 part[kLinkWaves][H];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int sub = wave % WPR, head = head_of<H>(lane);
    // The last rows first, eight workgroups at a time (a row stays on the XCD that the backward takes it to): they are what
    // the producer of the scores wrote last, and the first rows, which the backward starts with, are the last that passed
    // the memory-side cache.  Behind the copy that lays the scores out, that copy included, us, first rows first / last: B=64
    // L=512 H=8 float32 280.6 / 272.6, float16 219.7 / 218.3, B=16 L=1024 H=8 float16 219.5 / 217.2; the products that make
    // the scores and take the gradient, both copies, forward and backward together 1938 / 1935, 1135 / 1132, 1208 / 1206;
    // tensors that fit the cache: the same.
    const unsigned octet = gridDim.x & ~7u, blk = blockIdx.x < octet ? (octet - 8 - (blockIdx.x & ~7u)) + (blockIdx.x & 7u) : blockIdx.x;
    const int64_t row = (int64_t)blk * (kLinkWaves / WPR) + wave / WPR;
    if (row >= rows) { if (WPR > 1) __syncthreads(); return; }   // the one barrier of the others
    // The window is loaded before valid_end is known (up to the end of the row, which always exists), so
    // that a wave waits for one memory round trip, not two; what lies past valid_end is masked afterwards.
    const int i = (int)(row % L);
    const int nmax = L - 1 - i < translen ? L - 1 - i : translen;
    const TC *win = content + (row * L + i + 1) * H;
    float x[kLinkPer][H];
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k) {
        const int d = lane + (k * WPR + sub) * kWave;
        if (d < nmax) load_heads<TC, H>(win + (int64_t)d * H, x[k]);
    }
    const float gate2 = log_gates[row * H + head] * kLog2e;
    const LinkRow r = link_row(valid_end, row, L, translen);
    TC *out = links + row * translen;
    // Only the chunks that reach into the window are worked on (one wave-uniform test per chunk and pass: rows near the
    // end of a graph are short), and only the chunk that holds the end of the window needs masking.
    // per head: maximum, then the sum of exp(x - max) = 2^(x * log2e - max * log2e), over this wave's part of the window
    float m[H], sum[H];
#pragma unroll
    for (int c = 0; c < H; ++c) { m[c] = DAGX_NEG_INF; sum[c] = 0.f; }
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k) {
        const int d0 = (k * WPR + sub) * kWave;
        if (d0 < r.n) {
            if (d0 + kWave > r.n) {
                const bool in = lane + d0 < r.n;
#pragma unroll
                for (int c = 0; c < H; ++c) x[k][c] = in ? x[k][c] : DAGX_NEG_INF;
            }
#pragma unroll
            for (int c = 0; c < H; ++c) m[c] = fmaxf(m[c], x[k][c]);
        }
    }
    const float m_own = lanes_share<OpMax, H>(m, lane);
    lanes_spread<H>(m_own > DAGX_NEG_INF ? -m_own * kLog2e : 0.f, m);   // 0 for a head without any finite score: 2^(-inf) = 0, no NaN
    // the scores become e = 2^(x * log2e - max * log2e): their only exponential
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k)
        if ((k * WPR + sub) * kWave < r.n)
#pragma unroll
            for (int c = 0; c < H; ++c) { x[k][c] = fast_exp2(__builtin_fmaf(x[k][c], kLog2e, m[c])); sum[c] += x[k][c]; }
    float top = m_own, tot = lanes_share<OpSum, H>(sum, lane);
    if (WPR > 1) {
        if (lane < 16) part[wave][head] = make_float2(top, tot);
        __syncthreads();
        const int w0 = wave - sub;
        float2 q[WPR];
#pragma unroll
        for (int w = 0; w < WPR; ++w) { q[w] = part[w0 + w][head]; top = fmaxf(top, q[w].x); }
        tot = 0.f;
#pragma unroll
        for (int w = 0; w < WPR; ++w) tot += q[w].x > DAGX_NEG_INF ? q[w].y * fast_exp2((q[w].x - top) * kLog2e) : q[w].y;
    }
    // (a head without any finite score drops out; from here on every lane has the values of its head)
    const float log_tot = fast_log2(tot);
    const float lse2 = top > DAGX_NEG_INF ? __builtin_fmaf(top, kLog2e, log_tot) : DAGX_NEG_INF;
    const bool alive = lse2 > DAGX_NEG_INF;
    if (lse_out && sub == 0 && lane < 16) lse_out[row * H + head] = lse2 * kLn2;
    // mix the heads: log2 sum_c e_c * f_c with f = 2^(max - lse + gate), lane-local
    float f[H];
    const float f_own = alive && m_own > DAGX_NEG_INF ? fast_exp2(__builtin_fmaf(m_own - top, kLog2e, gate2 - log_tot)) : 0.f;
    lanes_spread<H>(f_own, f);
    const float bias_own = alive ? gate2 - lse2 : DAGX_NEG_INF, least = least_sum<H>(f_own, f);
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k) {
        const int d0 = (k * WPR + sub) * kWave, d = lane + d0;
        if (d0 >= translen) break;
        float v = DAGX_NEG_INF;
        if (d0 < r.n) {
            float acc = 0.f;
#pragma unroll
            for (int c = 0; c < H; ++c) acc = __builtin_fmaf(x[k][c], f[c], acc);
            const bool slow = d < r.n && !(acc >= least && acc <= kLinkHuge);
            if (d < r.n) v = fast_log2(acc) * kLn2;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(slow) != 0, 0)) {   // from the scores again, against the largest term
                float bias[H];
                lanes_spread<H>(bias_own, bias);
                if (slow) {
                    float y[H], ym = DAGX_NEG_INF;
                    load_heads<TC, H>(win + (int64_t)d * H, y);
#pragma unroll
                    for (int c = 0; c < H; ++c) { y[c] = __builtin_fmaf(y[c], kLog2e, bias[c]); ym = fmaxf(ym, y[c]); }
                    v = DAGX_NEG_INF;
                    if (ym > DAGX_NEG_INF) {
                        const float shift = ym < -DAGX_NEG_INF ? ym : 0.f;   // (a gate of +inf: the link is +inf, not inf - inf)
                        float acc2 = 0.f;
#pragma unroll
                        for (int c = 0; c < H; ++c) acc2 += fast_exp2(y[c] - shift);
                        v = (shift + fast_log2(acc2)) * kLn2;
                    }
                }
            }
        }
        if (d < translen) out[d] = from_float<TC>(v);
    }
}

// In place: content[b][i][j][c] <- d loss / d content, 0 outside the window; grad_gates[b][i][c] =
// d loss / d log_gates.  With p = exp(x - lse_c), G_c = exp(g_c) and q_c = grad_links[d] * G_c / sum_c' p_c' G_c':
//   d/dg_c = W_c = sum_d q[d][c] p[d][c],      d/dx[d][c] = p[d][c] * (q[d][c] - W_c):
// one exponential per score.  The normaliser over the heads is formed again from the scores, in float32, and not taken
// from the stored `links` (which the kernel does not read): rounded to bfloat16 a link value of -6 is 0.03 off, and every
// weight of its position with it by 3 %.
template <typename TC, int H, int WPR>
__global__ __launch_bounds__(kLinkThreads) void links_bwd_kernel(
    TC *__restrict__ content, const float *__restrict__ log_gates, const int64_t *__restrict__ valid_end,
    int64_t rows, int L, int translen, const float *__restrict__ lse_in,
    const TC *__restrict__ grad_links, float *__restrict__ grad_gates, bool past_caches) {
    __shared__ float part[kLinkWaves][H];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int sub = wave % WPR, head = head_of<H>(lane);
    const int64_t row = (int64_t)blockIdx.x * (kLinkWaves / WPR) + wave / WPR;
    if (row >= rows) { if (WPR > 1) __syncthreads(); return; }   // the one barrier of the others
    const int i = (int)(row % L);
    const int nmax = L - 1 - i < translen ? L - 1 - i : translen;
    TC *full = content + row * L * H;
    TC *win = full + (int64_t)(i + 1) * H;
    float x[kLinkPer][H], go[kLinkPer];   // scores, then p; incoming gradient, then grad / sum_c p_c G_c
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k) {
        const int d = lane + (k * WPR + sub) * kWave;
        if (d < nmax) {
            load_heads<TC, H>(win + (int64_t)d * H, x[k]);
            go[k] = to_float(grad_links[row * translen + d]);
        }
    }
    const float lse_own = lse_in[row * H + head], gate_own = log_gates[row * H + head];
    const LinkRow r = link_row(valid_end, row, L, translen);
    // outside the window: zeros (nothing of it is used), in contiguous pieces that pass the caches by if told to
    {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        using Piece = std::conditional_t<(sizeof(TC) * H >= 16), u32x4, u32x2>;
        constexpr int kEach = (int)(sizeof(TC) * H / sizeof(Piece));   // pieces per node
        Piece *p = reinterpret_cast<Piece *>(full);
        const int before = r.jlo * kEach, behind = (r.jlo + r.n) * kEach, end = L * kEach;
        const Piece zero = {};
        if (past_caches) {
            for (int q = lane + sub * kWave; q < before && q < end; q += WPR * kWave) __builtin_nontemporal_store(zero, p + q);
            for (int q = behind + lane + sub * kWave; q < end; q += WPR * kWave) __builtin_nontemporal_store(zero, p + q);
        } else {
            for (int q = lane + sub * kWave; q < before && q < end; q += WPR * kWave) p[q] = zero;
            for (int q = behind + lane + sub * kWave; q < end; q += WPR * kWave) p[q] = zero;
        }
    }
    const bool alive = lse_own > DAGX_NEG_INF;
    const bool every_head = __builtin_amdgcn_ballot_w64(alive) == ~0ull;
    float nlse[H], G[H], wsum[H];
    lanes_spread<H>(-lse_own * kLog2e, nlse);
    const float G_own = fast_exp2(gate_own * kLog2e);
    lanes_spread<H>(G_own, G);
    const float least = least_sum<H>(G_own, G);
    // The route of the positions whose sum or gradient leaves the range, and of rows with a head that reaches no position (or holds a
    // NaN, which reaches every gradient of the row): from the scores, against the largest term.  w: the position's d/dg_c,
    // pr: exp(x - lse).
    auto general = [&](int d, float grad, float (&w)[H], float (&pr)[H]) __attribute__((always_inline)) {
        float lse[H], gate[H], ym = DAGX_NEG_INF, acc = 0.f;
        lanes_spread<H>(lse_own, lse);
        lanes_spread<H>(gate_own, gate);
        load_heads<TC, H>(win + (int64_t)d * H, pr);
#pragma unroll
        for (int c = 0; c < H; ++c) {
            const float bias = lse[c] > DAGX_NEG_INF ? gate[c] - lse[c] : DAGX_NEG_INF;
            w[c] = (pr[c] + bias) * kLog2e;
            ym = fmaxf(ym, w[c]);
            pr[c] = (lse[c] > DAGX_NEG_INF && pr[c] > DAGX_NEG_INF) ? fast_exp2((pr[c] - lse[c]) * kLog2e) : 0.f;
        }
        const bool some = ym > DAGX_NEG_INF;   // else no head reaches this position: the weights stay 0
#pragma unroll
        for (int c = 0; c < H; ++c) {
            w[c] = some ? fast_exp2(w[c] - ym) : 0.f;   // (0 for a head that does not reach it, NaN for a NaN)
            acc += w[c];
        }
        const float t = some ? grad / acc : 0.f;
#pragma unroll
        for (int c = 0; c < H; ++c) w[c] = some ? w[c] * t : 0.f;
    };
#pragma unroll
    for (int c = 0; c < H; ++c) wsum[c] = 0.f;
    unsigned slow = 0;   // bit k: position k takes the general route
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k) {
        const int d0 = (k * WPR + sub) * kWave, d = lane + d0;
        if (d0 < r.n) {
            const bool in = d < r.n;
            float acc = 0.f;
#pragma unroll
            for (int c = 0; c < H; ++c) {
                x[k][c] = fast_exp2(__builtin_fmaf(x[k][c], kLog2e, nlse[c]));
                acc = __builtin_fmaf(x[k][c], G[c], acc);
            }
            const float grad = go[k];
            const bool fine = every_head && acc >= least && acc <= kLinkHuge && fabsf(grad) <= kLinkMostGrad;
            go[k] = in && fine ? grad / acc : 0.f;
            if (in && fine) {
#pragma unroll
                for (int c = 0; c < H; ++c) wsum[c] = __builtin_fmaf(go[k] * G[c], x[k][c], wsum[c]);   // (0 + q p: rounded once)
            }
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(in && !fine) != 0, 0)) {
                float w[H], pr[H];
                const bool mine = in && !fine;
                general(mine ? d : 0, grad, w, pr);
                if (mine) {
                    slow |= 1u << k;
#pragma unroll
                    for (int c = 0; c < H; ++c) wsum[c] += w[c];
                }
            }
        }
    }
    float W_own = lanes_share<OpSum, H>(wsum, lane);
    if (WPR > 1) {
        if (lane < 16) part[wave][head] = W_own;
        __syncthreads();
        const int w0 = wave - sub;
        W_own = 0.f;
#pragma unroll
        for (int w = 0; w < WPR; ++w) W_own += part[w0 + w][head];
    }
    if (sub == 0 && lane < 16) grad_gates[row * H + head] = W_own;
    float W[H];
    lanes_spread<H>(W_own, W);
#pragma unroll
    for (int k = 0; k < kLinkPer; ++k) {
        const int d0 = (k * WPR + sub) * kWave, d = lane + d0;
        if (d0 >= r.n) break;
        float dx[H];
#pragma unroll
        for (int c = 0; c < H; ++c) dx[c] = x[k][c] * (go[k] * G[c] - W[c]);   // (the product as in W: a window of one position gives 0)
        if (__builtin_expect(__builtin_amdgcn_ballot_w64((slow >> k) & 1u) != 0, 0)) {
            const bool mine = (slow >> k) & 1u;
            const float grad = d < r.n ? to_float(grad_links[row * translen + d]) : 0.f;
            float w[H], pr[H];
            general(mine ? d : 0, grad, w, pr);
            if (mine) {
#pragma unroll
                for (int c = 0; c < H; ++c) dx[c] = w[c] - W[c] * pr[c];
            }
        }
        if (d < r.n) store_heads<TC, H>(win + (int64_t)d * H, dx);
    }
}

static int check_links(const void *content, int dtype, const void *log_gates, const void *valid_end, int B, int L, int H,
                       int translen, const char *who) {
    if (B < 0 || L < 1 || H < 1 || translen < 1) { set_error("%s: bad sizes B=%d L=%d H=%d translen=%d", who, B, L, H, translen); return DAGX_ERR_ARGUMENT; }
    if (dtype < DAGX_F32 || dtype > DAGX_BF16) { set_error("%s: unsupported dtype", who); return DAGX_ERR_ARGUMENT; }
    if (H != 4 && H != 8 && H != 16) { set_error("%s: %d heads (4, 8 and 16 are supported)", who, H); return DAGX_ERR_UNSUPPORTED; }
    if (L > 1024) { set_error("%s: graph size L=%d exceeds the supported 1024", who, L); return DAGX_ERR_UNSUPPORTED; }
    if ((int64_t)B * L > 0x7fffffffLL) { set_error("%s: B*L too large for one launch", who); return DAGX_ERR_UNSUPPORTED; }
    if (B > 0 && (!content || !log_gates || !valid_end)) { set_error("%s: null pointer argument", who); return DAGX_ERR_ARGUMENT; }
    return DAGX_OK;
}

// Waves per row: the fewest that hold the longest window at kLinkPer positions a lane.
template <typename TC, int H>
static int launch_links_fwd(const void *content, const float *log_gates, const int64_t *valid_end, int B, int L, int translen,
                            void *links, float *lse, hipStream_t st) {
    const int64_t rows = (int64_t)B * L;
    const int n = translen < L - 1 ? translen : L - 1;
#define DAGX_GO(WPR) hipLaunchKernelGGL((links_fwd_kernel<TC, H, WPR>), dim3((unsigned)((rows * WPR + kLinkWaves - 1) / kLinkWaves)), dim3(kLinkThreads), 0, st, \
                                        static_cast<const TC *>(content), log_gates, valid_end, rows, L, translen, static_cast<TC *>(links), lse)
    if (n <= kLinkPer * kWave) DAGX_GO(1); else if (n <= 2 * kLinkPer * kWave) DAGX_GO(2); else DAGX_GO(4);
#undef DAGX_GO
    return check_launch("links_fwd");
}
template <typename TC, int H>
static int launch_links_bwd(void *content, const float *log_gates, const int64_t *valid_end, int B, int L, int translen,
                            const float *lse, const void *grad_links, float *grad_gates, hipStream_t st) {
    const int64_t rows = (int64_t)B * L;
    const int n = translen < L - 1 ? translen : L - 1;
    // The zeros pass the caches by where the tensor and what else is in use leave them no room in the 256 MB memory-side
    // cache; where they do, the transposition or batched product that reads the gradient next finds them there.  Forward and
    // backward between the copy that lays the scores out and the one that takes the gradient, B = 16 ... 64, L=512 H=8
    // float32 (us, past the caches / through them): transitions of any length 128 MB 190 / 181, 160 MB 237 / 226,
    // 192 MB 284 / 285, 224 MB 334 / 343, 512 MB 780 / 791; at most 32: 128 MB 167 / 152, 192 MB 247 / 239, 256 MB 327 /
    // 342, 512 MB 645 / 682.  float16 and bfloat16 cross near 192 MB too.  (Forward behind backward in one storage: equal up to
    // 160 MB, 25 / 32 in favour of the caches at 128 MB and transitions of at most 32, 75 / 78 against them at 192 MB.)
    const bool past_caches = rows * L * H * (int64_t)sizeof(TC) > (176 << 20);
#define DAGX_GO(WPR) hipLaunchKernelGGL((links_bwd_kernel<TC, H, WPR>), dim3((unsigned)((rows * WPR + kLinkWaves - 1) / kLinkWaves)), dim3(kLinkThreads), 0, st, \
                                        static_cast<TC *>(content), log_gates, valid_end, rows, L, translen, lse,                                               \
                                        static_cast<const TC *>(grad_links), grad_gates, past_caches)
    if (n <= kLinkPer * kWave) DAGX_GO(1); else if (n <= 2 * kLinkPer * kWave) DAGX_GO(2); else DAGX_GO(4);
#undef DAGX_GO
    return check_launch("links_bwd");
}

}  // namespace dagx

using namespace dagx;

#define DAGX_LINKS_DISPATCH(CALL)                                                                      \
    switch (dtype) {                                                                                   \
        case DAGX_F32: return H == 4 ? CALL(float, 4) : H == 8 ? CALL(float, 8) : CALL(float, 16);     \
        case DAGX_F16: return H == 4 ? CALL(__half, 4) : H == 8 ? CALL(__half, 8) : CALL(__half, 16);  \
        default: return H == 4 ? CALL(bf16_t, 4) : H == 8 ? CALL(bf16_t, 8) : CALL(bf16_t, 16);        \
    }

extern "C" int dagx_links_fwd(const void *content, int dtype, const float *log_gates, const int64_t *valid_end,
                              int B, int L, int H, int translen, void *links, float *lse, void *stream) {
    int rc = check_links(content, dtype, log_gates, valid_end, B, L, H, translen, "dag_links_fwd");
    if (rc) return rc;
    if (B == 0) return DAGX_OK;
    if (!links) { set_error("dag_links_fwd: the output pointer is null"); return DAGX_ERR_ARGUMENT; }
    hipStream_t st = static_cast<hipStream_t>(stream);
#define CALL(T, HH) launch_links_fwd<T, HH>(content, log_gates, valid_end, B, L, translen, links, lse, st)
    DAGX_LINKS_DISPATCH(CALL)
#undef CALL
}

extern "C" int dagx_links_bwd(void *content_inout, int dtype, const float *log_gates, const int64_t *valid_end,
                              int B, int L, int H, int translen, const void *links, const float *lse,
                              const void *grad_links, float *grad_gates, void *stream) {
    int rc = check_links(content_inout, dtype, log_gates, valid_end, B, L, H, translen, "dag_links_bwd");
    if (rc) return rc;
    if (B == 0) return DAGX_OK;
    if (!lse || !grad_links || !grad_gates) { set_error("dag_links_bwd: a saved-state or output pointer is null"); return DAGX_ERR_ARGUMENT; }
    hipStream_t st = static_cast<hipStream_t>(stream);
#define CALL(T, HH) launch_links_bwd<T, HH>(content_inout, log_gates, valid_end, B, L, translen, lse, grad_links, grad_gates, st)
    DAGX_LINKS_DISPATCH(CALL)
#undef CALL
}
