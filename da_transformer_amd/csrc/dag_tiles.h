// Building blocks shared by the tile-resident sweep kernels (log-semiring loss, max-semiring
// alignment): tile geometry, the grouping of position blocks into a pipeline of workgroups, the maximum
// over a wave, agent-scope loads/stores and copies to LDS for the hand-over, exponentials with a shift.
#pragma once

#include "dagx_common.h"

namespace dagx {

constexpr int kBlk = 64;            // positions per block
constexpr int kMaxBlocksFast = 16;  // fast path: L <= 1024
constexpr int kMaxGroups = 11;      // workgroups of one sweep
constexpr int kTileWaves = 8;       // waves per workgroup in the tile sweeps
constexpr int kTilesPerWave = 3;    // register-resident tiles per wave
constexpr int kTileCap = kTileWaves * kTilesPerWave;
// Linear-domain numbers of the fast sweep carry a constant factor 2^kShift2 each (transition probabilities
// and exp(residual) alike), so that the fp32 exponent range is used on both sides of 1: a transition or a
// residual survives down to exp(-126) instead of exp(-87), their product down to exp(-165).  Sums of
// products stay below 2^(2 * 56 + 10) < 2^128.
constexpr int kShift2 = 56;                       // in log2 units (38.8 nats)
constexpr float kMinLogP = -87.0f - 38.8f;        // a finite transition below this has no normal number in the scaled linear domain
constexpr float kTinyStored = 1.17549435e-38f;    // 2^-126: the smallest number that domain holds (a factor of exp(-126) under its scale)
constexpr int kSpinLimit = 1 << 22;

struct Tile { float p[kBlk]; };

// Number of tiles of position block Jb: predecessor blocks I in [ilo, Jb]; W = blocks a transition can span.
__device__ __host__ __forceinline__ int tile_ilo(int Jb, int W) { return Jb > W ? Jb - W : 0; }

// Host: workgroups per sweep needed for graph size L, each with at most `most` position blocks (0 = the fast path does not
// apply).
inline int groups_needed(int L, int translen, int most) {
    const int NB = (L + kBlk - 1) / kBlk;
    if (NB > kMaxBlocksFast) return 0;
    const int W = (translen + kBlk - 1) / kBlk;
    int groups = 1, sum = 0, blocks = 0;
    for (int Jb = 0; Jb < NB; ++Jb) {
        int c = Jb - tile_ilo(Jb, W) + 1;
        if (c > kTileCap) return 0;
        if (sum + c > kTileCap || blocks == most) { ++groups; sum = blocks = 0; }
        sum += c; ++blocks;
    }
    return groups <= kMaxGroups ? groups : 0;
}

// ---- DPP lane reductions (no LDS traffic) ----------------------------------------------------
__device__ __forceinline__ float lane_bcast(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
// max over the 64 lanes, wave-uniform result: butterfly inside the 16-lane rows (each DPP op needs its source written two wait
// states earlier), then the row results are folded across rows with the two wave-level DPP broadcasts (row 0 -> 1, row 2 -> 3 via
// row_bcast:15; rows 0-1 -> rows 2-3 via row_bcast:31) and lane 63 holds the maximum.
__device__ __forceinline__ float wave64_max(float v) {
    float r;
    asm("s_nop 1\n\t"
        "v_max_f32_dpp %0, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
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
        : "=&v"(r) : "v"(v));
    return lane_bcast(r, 63);
}

// A wave-uniform value the compiler must take as new at this point: address arithmetic built on it
// stays inside the loop (as one add per use) instead of being hoisted into a vector register that
// then lives across the whole loop.
__device__ __forceinline__ int opaque_uniform(int x) { asm volatile("" : "+s"(x)); return x; }

template <typename X>
__device__ __forceinline__ X load_agent(const X *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename X>
__device__ __forceinline__ void store_agent(X *p, X v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Wait until every vector-memory operation of this wave has completed.  Written as the builtin, not as
// inline assembly: the compiler's own wait-count bookkeeping then knows that nothing is outstanding and
// adds no second wait (which would also cover the stores issued in between) where a loop-carried load
// destination is rewritten.  Encoding: vmcnt = 0, expcnt = 7 (no wait), lgkmcnt = 15 (no wait).
// The empty asm statements keep the compiler from moving memory operations across the wait.
__device__ __forceinline__ void wait_vmem_all() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" ::: "memory");
}

// Asynchronous copy global -> LDS, one element per lane ("LDS-direct" load): the element at
// gbase + voff (bytes, per lane) lands in the dword at LDS byte address lds_byte + 4 * lane (16-bit
// elements zero-extended).  The hardware counts it in vmcnt like any vector load and completes it in
// issue order with the other vector loads and stores of the wave, but the compiler's wait-count
// bookkeeping does not see it: the code that uses these must place its own s_waitcnt (wait_vmem_*)
// before the data is read, and must not rely on compiler-computed vmcnt(N > 0) waits for other loads
// while such copies are in flight.
// the address as a value the compiler knows to be wave-uniform (so that it is handed to the
// instruction in scalar registers)
__device__ __forceinline__ unsigned long long uniform_address(const void *p) {
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(v & 0xffffffffULL));
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma_dword(unsigned lds_byte, const void *gbase, unsigned voff) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" :: "v"(voff), "s"(uniform_address(gbase)), "s"(lds_byte) : "memory", "m0");
}
__device__ __forceinline__ void dma_dword_agent(unsigned lds_byte, const void *gbase, unsigned voff) {   // agent-scope (sc1) load
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1 sc1" :: "v"(voff), "s"(uniform_address(gbase)), "s"(lds_byte) : "memory", "m0");
}
__device__ __forceinline__ void dma_ushort(unsigned lds_byte, const void *gbase, unsigned voff) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_ushort %0, %1" :: "v"(voff), "s"(uniform_address(gbase)), "s"(lds_byte) : "memory", "m0");
}
// The same with the base address already in scalar registers (a value taken through uniform_address once).
__device__ __forceinline__ void dma_dword_agent_u(unsigned lds_byte, unsigned long long ubase, unsigned voff) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1 sc1" :: "v"(voff), "s"(ubase), "s"(lds_byte) : "memory", "m0");
}
// sixteen bytes a lane, to lds_byte + 16 * lane (the global address at least 4-byte aligned)
__device__ __forceinline__ void dma_dwordx4_agent_u(unsigned lds_byte, unsigned long long ubase, unsigned voff) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 sc1" :: "v"(voff), "s"(ubase), "s"(lds_byte) : "memory", "m0");
}
#pragma clang diagnostic pop
template <typename X> __device__ __forceinline__ void dma_elem(unsigned lds_byte, const X *gbase, unsigned voff);
template <> __device__ __forceinline__ void dma_elem<float>(unsigned lds_byte, const float *gbase, unsigned voff) { dma_dword(lds_byte, gbase, voff); }
template <> __device__ __forceinline__ void dma_elem<__half>(unsigned lds_byte, const __half *gbase, unsigned voff) { dma_ushort(lds_byte, gbase, voff); }
template <> __device__ __forceinline__ void dma_elem<bf16_t>(unsigned lds_byte, const bf16_t *gbase, unsigned voff) { dma_ushort(lds_byte, gbase, voff); }
// value of an element that dma_elem<X> left in an LDS dword
template <typename X> __device__ __forceinline__ float dma_decode(unsigned raw);
template <> __device__ __forceinline__ float dma_decode<float>(unsigned raw) { return __builtin_bit_cast(float, raw); }
template <> __device__ __forceinline__ float dma_decode<__half>(unsigned raw) { return __half2float(__builtin_bit_cast(__half, (unsigned short)raw)); }
template <> __device__ __forceinline__ float dma_decode<bf16_t>(unsigned raw) { return __builtin_bit_cast(float, raw << 16); }

// 2^(x + kShift2) with the rounding errors of the unshifted function: the shift goes through the exponent field
// (ldexp), not through the argument of v_exp_f32, where adding 56 would cost five bits of the fraction.
__device__ __forceinline__ float exp2_shifted(float x) {
    // (arguments below -115, results under 2^-59, take the shift inside the argument instead: v_exp_f32 alone
    //  would flush them, and their rounding no longer matters)
    const bool deep = x < -115.f;
    const float r = fast_exp2(deep ? x + (float)kShift2 : x);
    return deep ? r : __builtin_ldexpf(r, kShift2);
}
// The staged transitions of the wide (float64) sweeps carry 2^kShiftLinksWide instead: their products are formed
// in float64, so the whole range of normal float32 numbers lies under a transition of probability one --
// log-probabilities down to kMinLogPWide = -(126 + 127) ln 2, rounded up.  (Not the subnormals below it: a
// subnormal has lost bits of its fraction, a transition of -190 came out 8 % off, and both sweeps of a sample
// carried the same wrong number, so nothing flagged it.  A log-probability above 0 overflows; the sample then
// fails its check and goes to the log-domain kernel.)
constexpr int kShiftLinksWide = 127;
constexpr float kMinLogPWide = -175.0f;
template <int SHIFT>
__device__ __forceinline__ float exp2_shifted_by(float x) {
    if constexpr (SHIFT == kShift2) return exp2_shifted(x);
    const bool deep = x < -115.f;   // (through a lifted argument, so that v_exp_f32 has a normal result, and down again by ldexp, which keeps subnormals)
    const float r = fast_exp2(deep ? x + (float)(SHIFT + 24) : x);
    return __builtin_ldexpf(r, deep ? -24 : SHIFT);
}
template <int SHIFT> __device__ __forceinline__ constexpr float min_logp() { return SHIFT == kShift2 ? kMinLogP : kMinLogPWide; }
// `tiny`: what a finite transition too small for the linear domain becomes -- 0 in a sweep that must never
// overstate (a lower bound of every sum), kTinyStored in one that must never understate (an upper bound).
template <int SHIFT>
__device__ __forceinline__ float link_prob(float e, bool valid, float tiny) {
    if (!valid) return 0.f;                 // (a NaN stays a NaN)
    if (e <= min_logp<SHIFT>()) return e > DAGX_NEG_INF ? tiny : 0.f;
    return exp2_shifted_by<SHIFT>(e * kLog2e);
}

}  // namespace dagx
