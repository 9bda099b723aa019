// Omni decoder attention for head dim 128 on CDNA4: FP32 operands, causal within each packed
// record, ungated (metal/clef.metal:2055-2319: omni_attn_prep, omni_attention).
//
// The reference keeps the P.V accumulator as an FP32 hi/lo pair so that thousands of updates
// do not round into one component. Here the P.V sums are FP32 within a tile of 32 keys and FP64 across tiles.
//
// Both products run on the bf16 matrix cores with every FP32 operand split into three bf16 parts
// and six products per pair (split32.h). Bounds of the item loop, per 32-key tile and SIMD: 192
// matrix instructions of 16 cycles against 128 FP32 ones of 32 cycles and 128 FP64 ones of 64 for
// the same work before. At 16,344 tokens, 32 / 4 heads: 27.85 -> 11.38 ms in turn on one box, 54% of the cycles on the
// matrix cores at 2.04 GHz; relative error against float64 3.3e-7 -> 1.8e-7 (most of it the FP32 output's
// rounding: the scores take 5 full-size roundings instead of 32). Where the scores do not matter, the FP32 sums
// within a tile show: constant V over 200 random scores comes back within 0.5 x 2^-24 rms, with FP64 products 0.2.
//
// Workgroup: one wave per q head of a GQA group (nh / nkv waves), all on the same 16 query
// rows of one record, so one 32-key K/V tile in LDS serves the whole group.
//   S^T = K . Q^T      A = 16 keys x 32 dims of K (LDS), B = the wave's Q (registers).
//   O^T += V^T . P^T   A = 16 dims x 32 keys of V^T (LDS), B = P (registers); FP32 over the
//                      tile's 32 keys (the full-size terms last, one rounding), FP64 across tiles.
// The A rows are read in a permuted order (key / dim 8 (r / 4) + 4 t + r % 4 for row r of tile t of a
// pair), so that a lane's scores are 8 consecutive keys, the B operand of the P.V product, and
// its outputs runs of 8 dims.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "split32.h"

namespace clef_hip {
namespace omni {

constexpr int HD = 128;
constexpr int BQ = 16;                  // query rows per block (every wave of the group)
constexpr int BK = 32;                  // keys per LDS tile
constexpr int SLACK = 32;               // zero rows after each kv head's T rows

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) double f64x4;

struct PrepParams {
    const float *qkv;           // [T][(nh + 2 nkv) * 128]
    const float *q_norm, *k_norm;
    const int32_t *pos3;        // [T][3]
    const float *freq;          // [192]: f32 inverse frequencies, then FP64 hi, lo parts
    float *q_plane;             // [nh][T][128]
    float *k_plane, *v_plane;   // [nkv][kvT][128]
    uint32_t *status;
    int nh, nkv, T, kvT, rope_exact;
    float eps;
};

struct AttnParams {
    const float *q_plane, *k_plane, *v_plane;
    const int32_t *blocks;      // [n_blk][8] {q_row0, nq, q_pos0, k_row0, k_len, 0, record, 0}
    float *out;                 // [T][nh * 128]
    int nh, nkv, T, kvT, n_blk;
    float scale;
};

// Rotary angle pos * f reduced to [-pi, pi] in FP64 (f = hi + lo, the FP64 frequency): the
// product of an integer below 2^24 and f is exact to FP64 rounding, and the reduction by a
// two-part 2*pi leaves an error far below FP32's resolution of the reduced angle.
__device__ __forceinline__ float omni_angle_exact(int position, float hi, float lo) {
    const double a = (double)position * ((double)hi + (double)lo);
    const double k = rint(a * 0.15915494309189535);   // 1 / (2 pi)
    double r = fma(-k, 6.283185307179586, a);          // 2 pi, FP64 nearest
    r = fma(-k, 2.4492935982947064e-16, r);           // 2 pi - its FP64 nearest
    return (float)r;
}

// One (pass row, head) item per 32 lanes; lane holds dims lane + 32 j, so the rotary pairs
// (d, d + 64) of d = lane and lane + 32 sit in the lane. Items past the pass rows zero the
// kv planes' slack rows.
__global__ __launch_bounds__(256) void omni_prep_kernel(PrepParams p) {
    const int heads = p.nh + p.nkv;
    const long item = (long)blockIdx.x * 8 + (threadIdx.x >> 5);
    const int lane = threadIdx.x & 31;
    const long n_items = (long)(p.T + SLACK) * heads;
    if (item >= n_items) return;
    const int t = (int)(item / heads), h = (int)(item % heads);
    const bool query = h < p.nh;
    const int kh = h - p.nh;
    if (t >= p.T) {
        if (!query) {
            float *kd = p.k_plane + ((size_t)kh * p.kvT + t) * HD, *vd = p.v_plane + ((size_t)kh * p.kvT + t) * HD;
#pragma unroll
            for (int j = 0; j < 4; j++) { kd[lane + 32 * j] = 0.f; vd[lane + 32 * j] = 0.f; }
        }
        return;
    }
    const size_t row = (size_t)(p.nh + 2 * p.nkv) * HD;
    const float *src = p.qkv + (size_t)t * row + (size_t)h * HD;
    const float *w = query ? p.q_norm : p.k_norm;
    float x[4], ss = 0.f;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        x[j] = src[lane + 32 * j];
        bad |= !isfinite(x[j]);
        ss += x[j] * x[j];
    }
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 32);
    const float inv = 1.0f / sqrtf(ss / (float)HD + p.eps);
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = x[j] * inv * w[lane + 32 * j];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        // interleaved M-RoPE over 64 pairs: pair i turns by axis i % 3, the last 4 by axis 0
        const int pair = lane + 32 * j, axis = pair < 60 ? pair % 3 : 0;
        const int position = p.pos3[3 * (size_t)t + axis];
        const float ang = p.rope_exact ? omni_angle_exact(position, p.freq[64 + pair], p.freq[128 + pair])
                                       : (float)position * p.freq[pair];
        float s, c;
        sincosf(ang, &s, &c);
        const float lo = x[j], hi = x[j + 2];
        x[j] = lo * c - hi * s;
        x[j + 2] = hi * c + lo * s;
    }
    if (query) {
        float *dst = p.q_plane + ((size_t)h * p.T + t) * HD;
#pragma unroll
        for (int j = 0; j < 4; j++) { bad |= !isfinite(x[j]); dst[lane + 32 * j] = x[j]; }
    } else {
        const float *vs = p.qkv + (size_t)t * row + (size_t)(p.nh + p.nkv + kh) * HD;
        float *kd = p.k_plane + ((size_t)kh * p.kvT + t) * HD, *vd = p.v_plane + ((size_t)kh * p.kvT + t) * HD;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float v = vs[lane + 32 * j];
            bad |= !isfinite(x[j]) || !isfinite(v);
            kd[lane + 32 * j] = x[j];
            vd[lane + 32 * j] = v;
        }
    }
    // A softmax max can hide a non-finite input; it is reported on its own.
    if (bad) atomicOr(p.status, 2u);
}

// max over the four 16-lane rows of a wave (permlane swaps, VALU only); every lane gets it
__device__ __forceinline__ float xrow_max(float x) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float m = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

// The rows of `rows` (a bit each) of a wave's 16 in plain FP32 with FP64 sums, for rows whose Q or a key that they see
// holds an infinity, a NaN or a magnitude from 2^55 on (split_bad): FP32 and FP64
// matrix products of operands straight from the planes, 16 keys at a time from the record's first, so that a
// row's bits do not depend on the rows beside it. One infinity that all tokens see, 32 / 4 heads: 425 tokens
// 115 us (row by row in vector code 1,300), 2,000 tokens 0.74 ms (8.7).
//   S^T = K . Q^T      A = 16 keys x 4 dims, B = Q: lane (g, r16) holds dims 16 c + 4 g + e of row r16.
//   O^T += V^T . P^T   A = dims 64 m + 4 i + e x keys 4 g + v, B = P: O is dims 64 m + 16 v + 4 g + e of row r16.
__device__ __forceinline__ void omni_rows_plain(const AttnParams &p, unsigned rows, int q_row0, int q_pos0, int k_row0, int k_len, int h, int kh) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const bool mine = (rows >> r16) & 1;
    const int r = mine ? r16 : __builtin_ctz(rows);
    const float *kbase = p.k_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    const float *vbase = p.v_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    const float *qs = p.q_plane + ((size_t)h * p.T + q_row0 + r) * HD + 4 * g;
    f32x4 q[8];
#pragma unroll
    for (int c = 0; c < 8; c++) q[c] = *(const f32x4 *)(qs + 16 * c);
    // keys that the lane's row sees, and the most that one of `rows` does
    const int keys = min(k_len, q_pos0 + r + 1), last = min(k_len, q_pos0 + 32 - __builtin_clz(rows));
    f64x4 o[2][4];
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int e = 0; e < 4; e++) o[m][e] = f64x4{0.0, 0.0, 0.0, 0.0};
    float m_run = -INFINITY;
    double l_run = 0.0;
    for (int kb = 0; kb < last; kb += 16) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        // every load goes out before the products (the compiler would wait for each)
        const float *kr = kbase + (size_t)min(kb + r16, k_len - 1) * HD + 4 * g;
        f32x4 k[8], w[4][2];
#pragma unroll
        for (int c = 0; c < 8; c++) k[c] = *(const f32x4 *)(kr + 16 * c);
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int m = 0; m < 2; m++) w[v][m] = *(const f32x4 *)(vbase + (size_t)min(kb + 4 * g + v, k_len - 1) * HD + 4 * r16 + 64 * m);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 8; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c][e], q[c][e], s, 0, 0, 0);
        // s[v] is the score of key kb + 4g + v for row r16
        float x[4], mx = -INFINITY, rs = 0.f;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            x[v] = kb + 4 * g + v < keys ? s[v] * p.scale : -INFINITY;
            mx = fmaxf(mx, x[v]);
        }
        const float mn = fmaxf(m_run, xrow_max(mx));
        const float alpha = m_run == -INFINITY ? (mn == -INFINITY ? 1.f : 0.f) : expf(m_run - mn);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            x[v] = x[v] == -INFINITY ? 0.f : expf(x[v] - mn);
            rs += x[v];
        }
        m_run = mn;
        l_run = l_run * (double)alpha + (double)rs;
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[m][e] *= (double)alpha;
        // infinities and NaN of V stay out of the matrix products, whose other rows may not see their keys
        bool special = false;
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int m = 0; m < 2; m++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float a = w[v][m][e];
                    const bool fin = isfinite(a);
                    special |= !fin;
                    o[m][e] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)(fin ? a : 0.f), (double)x[v], o[m][e], 0, 0, 0);
                }
        if (__any(special)) {
#pragma unroll 1
            for (int j = 0; j < 16; j++) {
                const int from = (j >> 2) * 16 + r16;   // the lane that holds key kb + j of row r16
                float pj = 0.f;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float y = __shfl(x[v], from);
                    pj = (j & 3) == v ? y : pj;
                }
                const float *vr = vbase + (size_t)min(kb + j, k_len - 1) * HD + 4 * g;
#pragma unroll
                for (int m = 0; m < 2; m++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const f32x4 a = *(const f32x4 *)(vr + 64 * m + 16 * v);
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (!isfinite(a[e]) && kb + j < keys) o[m][e][v] = fma((double)pj, (double)a[e], o[m][e][v]);
                    }
            }
        }
    }
    double l_row = l_run;
    l_row += __shfl_xor(l_row, 16);
    l_row += __shfl_xor(l_row, 32);
    if (!mine) return;
    const double il = l_row > 0.0 ? 1.0 / l_row : 0.0;
    float *dst = p.out + (size_t)(q_row0 + r) * p.nh * HD + (size_t)h * HD + 4 * g;
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            f32x4 w;
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = (float)(o[m][e][v] * il);
            *(f32x4 *)(dst + 64 * m + 16 * v) = w;
        }
}

// Grid: one workgroup per (block, kv head, W heads of its group); wave w is head w of those.
//
// K and V tiles of 32 keys are split into their bf16 parts once per workgroup, on the way from
// HBM to LDS: each thread's loads go out one tile ahead into registers, are split
// and stored as three bf16 planes (K rows, V transposed). LDS bytes of buffer b: K planes at
// b BUF + 8 KB p, V^T planes at b BUF + KV + 8 KB p (p = h, m, l).
//
// A trip has two halves: the products (S(t), and P.V(t - 1): the P.V product lags one tile) and
// the VALU work (softmax of S(t), splits of coming tiles), each closed by a barrier. With W = 8 (two
// waves per SIMD, one workgroup per CU) waves 4-7 run half a trip behind waves 0-3, so that on
// each SIMD one wave's products face the other's VALU work; in step, both waves wanted the matrix
// cores and then both the VALU, and the times added up. That takes three buffers: V(t)
// stages K(t + 2) and V(t + 1) while the later waves still read K(t) and V(t - 1). Smaller
// groups keep one buffer, staged between the two barriers, so that several workgroups share a CU.
template <int W>
__global__ __launch_bounds__(64 * W, W == 4 ? 2 : 1) void omni_attn_kernel(AttnParams p) {
    constexpr bool PP = W == 8;                            // the two wave groups half a trip apart
    constexpr int NB = PP ? 3 : 1, AH = PP ? 1 : 0;        // buffers; tiles staged ahead
    constexpr int PL = BK * HD * 2;                        // bytes of one plane (8 KB)
    constexpr int KV = 3 * PL, BUF = 2 * KV;               // K planes, then V^T planes
    constexpr int NP = 8 / W;                              // 8-element pieces of K (and of V) per thread
    __shared__ __attribute__((aligned(16))) uint8_t smem[NB * BUF];
    const int n_parts = p.nh / p.nkv / W, kh = blockIdx.x % p.nkv, part = blockIdx.x / p.nkv % n_parts, bi = blockIdx.x / p.nkv / n_parts;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int h = (kh * n_parts + part) * W + wave;
    const int32_t *blk = p.blocks + 8 * bi;
    const int q_row0 = blk[0], nq = blk[1], q_pos0 = blk[2], k_row0 = blk[3], k_len = blk[4];
    const int n_tiles = (k_len + BK - 1) / BK;
    const bool q_valid = r16 < nq;
    const int qpos = q_pos0 + r16, whole = min(k_len, q_pos0 + 1);   // whole: keys that every row sees
    const float *kbase = p.k_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    const float *vbase = p.v_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    float amax = 0.f;
    const split32::Weights wt;

    // ---- tile staging. Piece e of a thread: K dims 8 c .. 8 c + 7 of one key, V keys
    // 8 kg .. 8 kg + 7 of one dim.
    float kr[NP][8], vr[NP][8];
    auto load_k = [&](int kb) {
#pragma unroll
        for (int e = 0; e < NP; e++) {
            const int i = tid + 64 * W * e, key = i >> 4, c = i & 15;
            const f32x4 *s = (const f32x4 *)(kbase + (size_t)(kb + key) * HD + 8 * c);
            const f32x4 a = s[0], b = s[1];
#pragma unroll
            for (int j = 0; j < 4; j++) { kr[e][j] = a[j]; kr[e][4 + j] = b[j]; }
        }
    };
    auto load_v = [&](int kb) {
#pragma unroll
        for (int e = 0; e < NP; e++) {
            const int i = tid + 64 * W * e, d = i & 127, kg = i >> 7;
            const float *s = vbase + (size_t)(kb + 8 * kg) * HD + d;
#pragma unroll
            for (int j = 0; j < 8; j++) vr[e][j] = s[j * HD];
        }
    };
    auto put = [&](uint8_t *dst, const split32::Parts &s) __attribute__((always_inline)) {
        *(bf16x8 *)dst = s.h;
        *(bf16x8 *)(dst + PL) = s.m;
        *(bf16x8 *)(dst + 2 * PL) = s.l;
    };
    // K chunk c of key 8a + 4t + b sits at position c ^ (4a + b): the 16 rows one operand read
    // touches then hit 16 distinct 16-byte slots.
    auto put_k = [&](uint8_t *buf) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NP; e++) {
            const int i = tid + 64 * W * e, key = i >> 4, c = i & 15;
            amax = split32::split_amax(amax, kr[e]);
            put(buf + key * (2 * HD) + ((c ^ ((key & 3) | ((key >> 3) << 2))) * 16), split32::split8(kr[e], wt));
        }
    };
    // V^T row d: its four 8-key chunks at position kg ^ (-(d / 8) % 4) ^ ((d / 4) % 2): the 16
    // lanes one step of a ds_read_b128 or ds_write_b128 serves, consecutive or {0-3, 12-15, 20-27}
    // and its like, hit 16 distinct 16-byte slots.
    auto put_v = [&](uint8_t *buf) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NP; e++) {
            const int i = tid + 64 * W * e, d = i & 127, kg = i >> 7;
            amax = split32::split_amax(amax, vr[e]);
            split32::scale_v(vr[e]);
            put(buf + KV + d * (2 * BK) + ((kg ^ (-(d >> 3) & 3) ^ ((d >> 2) & 1)) * 16), split32::split8(vr[e], wt));
        }
    };
    // Keys past the item's range (slack, or another record's) become zeros: their zero probabilities
    // then give zero products, and what lies there cannot send a row down the plain path. So do values of V
    // that are left to it, in tiles that some row sees in part.
    auto clear_k = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NP; e++)
#pragma unroll
            for (int j = 0; j < 8; j++) kr[e][j] = kb + ((tid + 64 * W * e) >> 4) < k_len ? kr[e][j] : 0.f;
    };
    auto clear_v = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NP; e++) {
            const int kg = (tid + 64 * W * e) >> 7;
#pragma unroll
            for (int j = 0; j < 8; j++) vr[e][j] = kb + 8 * kg + j < k_len ? vr[e][j] : 0.f;
            amax = split32::split_amax(amax, vr[e]);
#pragma unroll
            for (int j = 0; j < 8; j++) vr[e][j] = split32::split_bad(vr[e][j]) ? 0.f : vr[e][j];
        }
    };

    // ---- per-lane LDS byte addresses of the operand reads (plane h of buffer 0)
    const unsigned lds0 = split32::lds_offset(smem);
    unsigned ka[4];   // 32-dim step c: K row of S^T A row r16 in subtile 0 (subtile 1: + 4 rows)
#pragma unroll
    for (int c = 0; c < 4; c++) ka[c] = lds0 + (8 * (r16 >> 2) + (r16 & 3)) * (2 * HD) + (((4 * c + g) ^ r16) * 16);
    unsigned va[2];   // V^T row of O^T A row r16 in dim tiles 0 and 1 (tiles 2u + w: + 32 u rows)
#pragma unroll
    for (int w = 0; w < 2; w++)
        va[w] = lds0 + KV + (8 * (r16 >> 2) + 4 * w + (r16 & 3)) * (2 * BK) + ((g ^ (-(r16 >> 2) & 3) ^ w) * 16);

    if (n_tiles > 0) {
        load_k(0);
        load_v(0);
    }
    // ---- Q: lane holds Q[row r16][32 c + 8 g + j], the B operand of step c, scaled by
    // scale * log2 e (the scores then are exponents of 2)
    bf16x8 qh[4], qm[4], ql[4];
    {
        const float sl2 = p.scale * 1.4426950408889634f;
        const float *qs = p.q_plane + ((size_t)h * p.T + q_row0 + (q_valid ? r16 : 0)) * HD + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const f32x4 a = *(const f32x4 *)(qs + 32 * c), b = *(const f32x4 *)(qs + 32 * c + 4);
            float x[8];
#pragma unroll
            for (int j = 0; j < 4; j++) { x[j] = a[j] * sl2; x[4 + j] = b[j] * sl2; }
            amax = split32::split_amax(amax, x);
            const split32::Parts s = split32::split8(x, wt);
            qh[c] = s.h; qm[c] = s.m; ql[c] = s.l;
        }
    }
    // tile t's operands live in buffer t % NB; registers hold the tiles staged next
    if (n_tiles > 0) {
        if (BK > k_len) clear_k(0);
        put_k(smem);
        if (n_tiles > 1) load_k(BK);
        if constexpr (PP) {
            if (BK > whole) clear_v(0);
            put_v(smem);
            if (n_tiles > 1) {
                load_v(BK);
                if (2 * BK > k_len) clear_k(BK);
                put_k(smem + BUF);
                if (n_tiles > 2) load_k(2 * BK);
            }
        }
    }
    // every LDS access of the half trip is done; the loads in flight stay so
    auto half_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    half_barrier();

    f64x4 o[8];
#pragma unroll
    for (int n = 0; n < 8; n++) o[n] = f64x4{0.0, 0.0, 0.0, 0.0};
    // the running maximum starts at the lowest finite value: a row that has seen no key yet then
    // needs no case of its own (its probabilities are 2^-inf = 0)
    float m_run = -3.4028235e38f;
    double l_run = 0.0;
    bf16x8 ph, pm, pl;   // P of the previous tile

    // The products of a trip: S^T of the tile at kbuf (two 16-key subtiles, four 32-dim steps; the hh
    // terms in one accumulator, the smaller ones in another), and O^T += V^T . P^T of the tile at
    // vbuf (pairs of 16-dim tiles, FP32 over the tile's 32 keys, then into the FP64
    // accumulators). Every step is six operand reads and twelve products.
    auto products = [&](unsigned kbuf, unsigned vbuf, auto S, auto PV, float (&x)[8]) __attribute__((always_inline)) {
        constexpr int n_s = decltype(S)::value ? 4 : 0, n = n_s + (decltype(PV)::value ? 4 : 0);
        constexpr int LOOK = W == 4 ? 1 : 2;   // steps the reads run ahead (two waves of W = 4 share a SIMD's registers with 16 staged values more)
        split32::Six ring[LOOK];
        auto read = [&](auto I) {
            constexpr int i = decltype(I)::value;
            if constexpr (i < n_s) split32::read6<0, PL>(ring[i % LOOK], ka[i] + kbuf, ka[i] + kbuf + 4 * 2 * HD);
            else split32::read6<32 * (i - n_s) * 2 * BK, PL>(ring[i % LOOK], va[0] + vbuf, va[1] + vbuf);
        };
        f32x4 s[2], sx[2], acc[2][2];
#pragma unroll
        for (int u = 0; u < 2; u++) s[u] = sx[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        read(std::integral_constant<int, 0>{});
        if constexpr (LOOK > 1 && n > 1) read(std::integral_constant<int, 1>{});
        // what step i - 1 left to the VALU, in six parts between step i's products: placed right
        // after their own chain's end the sums would wait for it, and the products behind them
        auto rest = [&](auto I, auto J) {
            constexpr int i = decltype(I)::value, j = decltype(J)::value;
            if constexpr (i == n_s && n_s > 0) {
                if constexpr (j >= 2) {
#pragma unroll
                    for (int e = 2 * (j - 2); e < 2 * (j - 1); e++) x[e] = s[e >> 2][e & 3] + sx[e >> 2][e & 3];
                }
            } else if constexpr (i > n_s && j >= 2) {
                constexpr int k = i - 1 - n_s;
#pragma unroll
                for (int e = 2 * (j - 2); e < 2 * (j - 1); e++) o[2 * k + (e >> 2)][e & 3] += (double)acc[k & 1][e >> 2][e & 3];
            }
        };
        split32::sfor<n>([&](auto I) {
            constexpr int i = decltype(I)::value;
            split32::wait6<(LOOK > 1 && i + 1 < n ? 6 : 0)>(ring[i % LOOK]);
            const split32::Six a = ring[i % LOOK];
            if constexpr (i < n_s) {
                split32::mma6_apart(s, sx, a, qh[i], qm[i], ql[i]);
            } else {
                constexpr int k = i - n_s;
                f32x4(&c)[2] = acc[k & 1];
                c[0] = c[1] = f32x4{0.f, 0.f, 0.f, 0.f};
                __builtin_amdgcn_sched_barrier(0);
                split32::sfor<6>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    split32::mma6_term<j>(c[0], c[1], a, ph, pm, pl);
                    rest(I, J);
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
            if constexpr (i + LOOK < n) read(std::integral_constant<int, i + LOOK>{});
        });
        if constexpr (n > n_s) {
#pragma unroll
            for (int e = 0; e < 8; e++) o[6 + (e >> 2)][e & 3] += (double)acc[1][e >> 2][e & 3];
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = s[e >> 2][e & 3] + sx[e >> 2][e & 3];
        }
    };
    // One trip (FIRST: no P.V yet). EDGE: some key of the tile lies past a row's position, or the
    // tiles it stages may reach past the record's end.
    int bt = 0;   // t % NB
    auto trip = [&](const int t, auto FIRST, auto EDGE) __attribute__((always_inline)) {
        constexpr bool first = decltype(FIRST)::value, edge = decltype(EDGE)::value;
        const int kb = t * BK;
        const int b_next = bt + 1 < NB ? bt + 1 : 0, b_prev = bt > 0 ? bt - 1 : NB - 1;
        float x[8];
        // the wave in its products goes first where both of a SIMD's waves want to issue (2.5% at
        // 16,344 tokens; the other way round 1% slower)
        if constexpr (PP) __builtin_amdgcn_s_setprio(1);
        products(bt * BUF, b_prev * BUF, std::true_type{}, std::integral_constant<bool, !first>{}, x);
        if constexpr (PP) __builtin_amdgcn_s_setprio(0);
        half_barrier();
        // stage K(t + 1 + AH) and V(t + AH), then load the tiles after them
        if (!edge || t + 1 + AH < n_tiles) {
            if (edge && kb + (2 + AH) * BK > k_len) clear_k(kb + (1 + AH) * BK);
            put_k(smem + (PP ? b_prev : 0) * BUF);
        }
        if (!edge || t + 2 + AH < n_tiles) load_k(min(t + 2 + AH, n_tiles - 1) * BK);
        if (!edge || t + AH < n_tiles) {
            if (edge && kb + (1 + AH) * BK > whole) clear_v(kb + AH * BK);
            put_v(smem + (PP ? b_next : 0) * BUF);
        }
        if (!edge || t + 1 + AH < n_tiles) load_v(min(t + 1 + AH, n_tiles - 1) * BK);
        // x[4 u + v] is the score (exponent of 2) of key kb + 8g + 4u + v for row r16
        if constexpr (edge) {
            const int lim = min(k_len - 1, qpos) - kb - 8 * g;
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = j <= lim ? x[j] : -INFINITY;
        }
        float mx = x[0];
#pragma unroll
        for (int j = 1; j < 8; j++) mx = fmaxf(mx, x[j]);
        const float mn = fmaxf(m_run, xrow_max(mx));
        const float alpha = __builtin_amdgcn_exp2f(m_run - mn);
        float rs = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            x[j] = split32::P_SCALE * __builtin_amdgcn_exp2f(x[j] - mn);   // a masked key's -inf gives 0
            rs += x[j];
        }
        m_run = mn;
        l_run = l_run * (double)alpha + (double)rs;
        const split32::Parts pp = split32::split8(x, wt);
        ph = pp.h; pm = pp.m; pl = pp.l;
        if constexpr (!first) {
            if (__any(alpha != 1.f)) {
                // in place (as plain C++ the other path of this branch copied all 64 registers)
                const double ad = (double)alpha;
#pragma unroll
                for (int n = 0; n < 8; n++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        double d = o[n][v];
                        asm("v_mul_f64 %0, %0, %1" : "+v"(d) : "v"(ad));
                        o[n][v] = d;
                    }
            }
        }
        half_barrier();
        bt = b_next;
    };
    using T = std::true_type;
    using F = std::false_type;
    // trips whose tile every row sees whole, as the V that they stage, with the K they stage inside the record
    const int n_inner = min((q_pos0 + 1) / BK - AH, k_len / BK - AH - 1);
    if (n_tiles > 0) {
        const bool late = PP && wave >= W / 2;
        if (late) half_barrier();
        int t = 0;
        if (n_inner > 0) trip(t++, T{}, F{});
        else trip(t++, T{}, T{});
        for (; t < n_inner; t++) trip(t, F{}, F{});
        for (; t < n_tiles; t++) trip(t, F{}, T{});
        if (PP && !late) half_barrier();
        float none[8];
        products(0, (bt > 0 ? bt - 1 : NB - 1) * BUF, F{}, T{}, none);
    }

    // ---- epilogue: O = O^T / l; lane holds dims 32 u + 8 g + 4 w + v of row r16 (tile 2u + w, entry v)
    double l_row = l_run;
    l_row += __shfl_xor(l_row, 16);
    l_row += __shfl_xor(l_row, 32);
    bool plain = false;
    if (__syncthreads_or(!split32::split_fine(amax))) {
        const int first = split32::first_bad_key<HD>(kbase, vbase, k_len, (int *)smem);
        int own = 0;
#pragma unroll
        for (int c = 0; c < 4; c++) own |= split32::query_bad(qh[c]);
        own |= __shfl_xor(own, 16);
        own |= __shfl_xor(own, 32);
        plain = q_valid && (own || first <= qpos);
    }
    if (q_valid && !plain) {
        const double il = l_row > 0.0 ? (1.0 / split32::V_SCALE) / l_row : 0.0;
        float *dst = p.out + (size_t)(q_row0 + r16) * p.nh * HD + (size_t)h * HD + 8 * g;
#pragma unroll
        for (int n = 0; n < 8; n++) {
            f32x4 w;
#pragma unroll
            for (int v = 0; v < 4; v++) w[v] = (float)(o[n][v] * il);
            *(f32x4 *)(dst + 32 * (n >> 1) + 4 * (n & 1)) = w;
        }
    }
    const unsigned rows = (unsigned)__ballot(plain) & 0xffffu;
    if (rows) omni_rows_plain(p, rows, q_row0, q_pos0, k_row0, k_len, h, kh);
}

}  // namespace omni
}  // namespace clef_hip
