// FP32 products on the bf16 matrix cores of CDNA4 (gfx950).
//
// An FP32 value is the exact sum of three bf16 values: h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m), each rounded to nearest even, so |m| <= 2^-8 |x| and |l| <= 2^-17 |x|. A product a . b then
// takes the six terms hh, hm, mh, hl, lh, mm; the three left out (ml, lm, ll) are at most 2^-24 |a b| together, the
// rounding of one FP32 product (2^-27 |a b| root mean square over random operands). The terms run on v_mfma_f32_16x16x32_bf16 with FP32
// accumulation, the small ones first or into accumulators of their own, so that the full-size sum
// is rounded once per 32-deep step, where v_mfma_f32_16x16x4f32 rounds it once per 4: the score of 256 equal operands
// 0x1.00ff8p+0, whose left-out terms all have one sign, is off by 0.1 x 2^-24, with the FP32 instruction by 16. Six bf16
// products cost 6 / 16 of the FP32 matrix instructions' time (2.5 PFLOP/s against 157 TFLOP/s).
//
// The split is exact for finite |x| below bf16's overflow threshold (0x7f7f8000) down to 2^-110; smaller values lose
// what lies below 2^-133, bf16's smallest subnormal. V and P are split as 2^24 times their value, which every FP32
// value survives whole (their products go into a sum that may be as small as they are; unscaled, values of
// 1e-35 came back with an error of 2^-19, and below 2^-134 as zeros; the multiplications cost 1% of C1 in FP32, 3%
// of a 425-token pass, 2% of Omni's 16,344). Q and K need no scale: what a product of theirs loses is below 2^-133 x
// 2^55 (LIMIT) = 2^-78 of a score.
#pragma once
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include <utility>

#include "bf16_ops.h"

namespace clef_hip {
namespace split32 {

typedef __attribute__((ext_vector_type(4))) float f32x4;

// The parts of eight consecutive contraction elements: one 16x16x32 operand each.
struct Parts {
    bf16x8 h, m, l;
};

// x - h of one element of a packed pair: v_dot2_f32_bf16 with weights (-1, 0) or (0, -1), one instruction
// for the widening and the subtraction. The difference is exact, so the instruction's own rounding does not
// enter (a value that passes through the attention kernels alone comes back bit for bit, over all exponents:
// tests/test_gpu_fp32.py). The weights sit in
// registers the compiler cannot see through: as constants it encoded (-1, 0) wrongly.
struct Weights {
    unsigned lo, hi;
    __device__ __forceinline__ Weights() : lo(0x0000bf80u), hi(0xbf800000u) { asm("" : "+s"(lo), "+s"(hi)); }
};
__device__ __forceinline__ float minus_lo(unsigned pair, const Weights &w, float x) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, w.lo), x, false);
}
__device__ __forceinline__ float minus_hi(unsigned pair, const Weights &w, float x) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, w.hi), x, false);
}

// Part by part over the eight elements: pair by pair, each conversion waited for the differences ahead of it
// (C1 FP32 303 -> 296 us, Omni 1 - 3%).
__device__ __forceinline__ Parts split8(const float (&x)[8], const Weights &w) {
    u32x4 h, m, l;
    float r[8];
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = pack_bf16(x[2 * i], x[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 4; i++) { r[2 * i] = minus_lo(h[i], w, x[2 * i]); r[2 * i + 1] = minus_hi(h[i], w, x[2 * i + 1]); }
#pragma unroll
    for (int i = 0; i < 4; i++) m[i] = pack_bf16(r[2 * i], r[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 4; i++) { r[2 * i] = minus_lo(m[i], w, r[2 * i]); r[2 * i + 1] = minus_hi(m[i], w, r[2 * i + 1]); }
#pragma unroll
    for (int i = 0; i < 4; i++) l[i] = pack_bf16(r[2 * i], r[2 * i + 1]);
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

// Values that are left to plain arithmetic: infinities, NaN and magnitudes from 2^55 on. Below, no score overflows
// (256 products of 2^110), nor does a sum of V: 2^55 x 2^24 x 2^24 (the scales) in each of up to 2^24 keys.
// A row is computed with plain arithmetic if its own Q or a key that it sees holds such a value, which does
// not depend on how the pass is cut into items. A kernel therefore
//   keeps the largest magnitude it splits (split_amax); an item without such values (split_fine) is done;
//   stages such values of V as zeros in tiles that some row sees in part, so that the rows which do not see
//     them keep their sums, with that key's zero probability, clear of infinities and NaN;
//   finds the first key with such a value (first_bad_key) and the rows concerned at an item's end.
constexpr float LIMIT = 0x1p55f, V_SCALE = 0x1p24f, P_SCALE = 0x1p24f;   // the output's 1 / l divides by V_SCALE, P's is in l
__device__ __forceinline__ bool split_bad(float x) { return !(fabsf(x) < LIMIT); }
// Largest magnitude of a running maximum and eight values; a NaN stays. (In asm: with the builtin the
// compiler kept the values longer and spilled 13 registers of the text kernel.)
__device__ __forceinline__ float split_amax(float amax, const float (&x)[8]) {
    asm("v_maximum3_f32 %0, |%1|, |%2|, %0\n\tv_maximum3_f32 %0, |%3|, |%4|, %0\n\t"
        "v_maximum3_f32 %0, |%5|, |%6|, %0\n\tv_maximum3_f32 %0, |%7|, |%8|, %0"
        : "+&v"(amax) : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]));
    return amax;
}
// (the margin: a bad query is told by its high parts, rounded)
__device__ __forceinline__ bool split_fine(float amax) { return amax < 0.99f * LIMIT; }
__device__ __forceinline__ bool query_bad(bf16x8 h) {
    const u32x4 w = __builtin_bit_cast(u32x4, h);
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; i++) bad |= split_bad(bf_lo(w[i])) || split_bad(bf_hi(w[i]));
    return bad;
}
// The first of k_len keys with such a value in its K or V row (HD dims, rows HD apart), INT_MAX: none. Every thread
// of the workgroup calls it; `shared` is an LDS word that nobody uses any more.
template <int HD>
__device__ __forceinline__ int first_bad_key(const float *k, const float *v, int k_len, int *shared) {
    const int per_row = HD / 4, c = threadIdx.x % per_row * 4;
    __syncthreads();
    if (threadIdx.x == 0) *shared = INT_MAX;
    __syncthreads();
    for (int key = threadIdx.x / per_row; key < k_len && key < *(volatile int *)shared; key += blockDim.x / per_row) {
        const f32x4 a = *(const f32x4 *)(k + (size_t)key * HD + c), b = *(const f32x4 *)(v + (size_t)key * HD + c);
        bool bad = false;
        for (int e = 0; e < 4; e++) bad |= split_bad(a[e]) || split_bad(b[e]);
        if (bad) atomicMin(shared, key);
    }
    __syncthreads();
    return *shared;
}

__device__ __forceinline__ void scale_v(float (&x)[8]) {
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] *= V_SCALE;
}

template <typename F, int... I>
__device__ __forceinline__ void sfor_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void sfor(F &&f) {
    sfor_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ unsigned lds_offset(const void *p) { return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void *)p; }

// Operand reads two steps ahead of their products, for kernels with the registers for it: six
// ds_read_b128 (the h, m, l parts of two operands) as one asm statement, and a wait that names them.
struct Six {
    bf16x8 h0, m0, l0, h1, m1, l1;
};
// operands at a + O and b + O, their parts PL bytes apart
template <int O, int PL>
__device__ __forceinline__ void read6(Six &r, unsigned a, unsigned b) {
    asm volatile("ds_read_b128 %0, %6 offset:%8\n\tds_read_b128 %3, %7 offset:%8\n\t"
                 "ds_read_b128 %1, %6 offset:%9\n\tds_read_b128 %4, %7 offset:%9\n\t"
                 "ds_read_b128 %2, %6 offset:%10\n\tds_read_b128 %5, %7 offset:%10"
                 : "=&v"(r.h0), "=&v"(r.m0), "=&v"(r.l0), "=&v"(r.h1), "=&v"(r.m1), "=&v"(r.l1)
                 : "v"(a), "v"(b), "i"(O), "i"(O + PL), "i"(O + 2 * PL) : "memory");
}
template <int N>   // until at most N LDS operations are outstanding
__device__ __forceinline__ void wait6(Six &r) {
    asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(r.h0), "+v"(r.m0), "+v"(r.l0), "+v"(r.h1), "+v"(r.m1), "+v"(r.l1) : "i"(N) : "memory");
}

// Two products of split operands against one split operand: hh into big, the five smaller terms
// into small (the caller may pass one accumulator for both: the small terms then come first).
__device__ __forceinline__ void mma6_apart(f32x4 (&big)[2], f32x4 (&small)[2], const Six &a, bf16x8 bh, bf16x8 bm, bf16x8 bl) {
    small[0] = mma(a.l0, bh, small[0]);
    small[1] = mma(a.l1, bh, small[1]);
    big[0] = mma(a.h0, bh, big[0]);
    big[1] = mma(a.h1, bh, big[1]);
    small[0] = mma(a.h0, bl, small[0]);
    small[1] = mma(a.h1, bl, small[1]);
    small[0] = mma(a.m0, bm, small[0]);
    small[1] = mma(a.m1, bm, small[1]);
    small[0] = mma(a.m0, bh, small[0]);
    small[1] = mma(a.m1, bh, small[1]);
    small[0] = mma(a.h0, bm, small[0]);
    small[1] = mma(a.h1, bm, small[1]);
}
// term j of the six, smallest first, of two products into one accumulator each
template <int J>
__device__ __forceinline__ void mma6_term(f32x4 &c0, f32x4 &c1, const Six &a, bf16x8 bh, bf16x8 bm, bf16x8 bl) {
    constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};   // parts: 0 h, 1 m, 2 l
    const bf16x8 b = B[J] == 0 ? bh : B[J] == 1 ? bm : bl;
    c0 = mma(A[J] == 0 ? a.h0 : A[J] == 1 ? a.m0 : a.l0, b, c0);
    c1 = mma(A[J] == 0 ? a.h1 : A[J] == 1 ? a.m1 : a.l1, b, c1);
}

// Products of a pair of 16-row A operands (two 16-key subtiles of K, two 16-dim tiles of V^T) with
// one B operand: six ds_read_b128 and twelve products a step, as a stream whose reads roll one step
// ahead through the same 24 registers: a part's two registers take the next step's read as soon as their
// last product has issued. Reads, waits and products come in the order l, m, h, so that at each wait the four
// newest reads may stay in flight.
template <int OA, int OB>
__device__ __forceinline__ void read_pair(bf16x8 (&r)[2], unsigned a, unsigned b) {
    static_assert(OA < 65536 && OB < 65536, "16-bit offsets");
    asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%5"
                 : "=&v"(r[0]), "=&v"(r[1]) : "v"(a), "v"(b), "i"(OA), "i"(OB) : "memory");
}
template <int N>   // until at most N LDS operations are outstanding
__device__ __forceinline__ void wait_pair(bf16x8 (&r)[2]) {
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(r[0]), "+v"(r[1]) : "i"(N) : "memory");
}
struct Ring {
    bf16x8 l[2], m[2], h[2];
};
// AT: OA, OB (byte offsets of the two operands' h parts) and the addresses they add to; the m and l
// parts lie PL and 2 PL behind.
template <int PL, int OA, int OB>
__device__ __forceinline__ void ring_start(Ring &r, unsigned a, unsigned b) {
    read_pair<OA + 2 * PL, OB + 2 * PL>(r.l, a, b);
    read_pair<OA + PL, OB + PL>(r.m, a, b);
    read_pair<OA, OB>(r.h, a, b);
}
// One step: the products of the operands in the ring with (bh, bm, bl), hh into big and the smaller terms into
// small (which may be the same accumulators), and the reads of the next step's operands
// (MORE) at OA, OB.
template <int PL, bool MORE, int OA, int OB>
__device__ __forceinline__ void ring_step(Ring &r, unsigned a, unsigned b, f32x4 &big0, f32x4 &big1, f32x4 &small0, f32x4 &small1,
                                          bf16x8 bh, bf16x8 bm, bf16x8 bl) {
    auto pair = [&](const bf16x8 (&x)[2], bf16x8 y, f32x4 &c0, f32x4 &c1) {
        c0 = mma(x[0], y, c0);
        c1 = mma(x[1], y, c1);
    };
    wait_pair<4>(r.l);
    pair(r.l, bh, small0, small1);
    if constexpr (MORE) read_pair<OA + 2 * PL, OB + 2 * PL>(r.l, a, b);
    wait_pair<(MORE ? 4 : 2)>(r.m);
    pair(r.m, bm, small0, small1);
    pair(r.m, bh, small0, small1);
    if constexpr (MORE) read_pair<OA + PL, OB + PL>(r.m, a, b);
    wait_pair<(MORE ? 4 : 0)>(r.h);
    pair(r.h, bl, small0, small1);
    pair(r.h, bm, small0, small1);
    pair(r.h, bh, big0, big1);
    if constexpr (MORE) read_pair<OA, OB>(r.h, a, b);
}

}  // namespace split32
}  // namespace clef_hip
