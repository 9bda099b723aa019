// FP32 text attention for head dim 256 on CDNA4 (gfx950): the precision the reference's FP32
// kernels give (metal/clef.metal:250-302 attn_prep, 316-654 attention / attention_fa /
// attention_reuse / attention_prefetch_64), used for the per-record rerun after an f16 overflow
// (clef.c:526-550) and with CLEF_ATTN_TU=0.
//
// Semantics (the reference's, per query row t of head h, kv head h / (nh / nkv)):
//   q, k = RMSNorm(x) * w (w as given, already 1 + w), then partial rotary over dims [0, 64):
//   pair (i, i + 32) turns by pos3[t][i % 3] * inv_freq[i]; V copied. S = (q . k) * scale over
//   the record's keys up to the query's position, softmax with exp, O = P.V / l, times
//   sigmoid(gate) (the second half of the head's row), written through act16 (bf16, or f16
//   that saturates and flags the record) or as f32.
//
// Everything is held in FP32; the products run on the bf16 matrix cores with every operand split
// into three bf16 parts and six products per pair (split32.h), FP32 accumulation, the softmax in FP32
// VALU (exp2 domain). Key tiles start at the record's first key, so a record's arithmetic does not
// depend on what is packed with it.
//
// Workgroup: NW waves of 16 query rows, R row groups x k heads of one kv group (f32_shape), so one
// 32-key K / V tile in LDS (three bf16 planes each, 96 KB) serves up to 128 rows.
//   S^T = K . Q^T      A = 16 keys x 32 dims of K (LDS), B = the wave's Q (registers, 96 of them).
//   O^T += V^T . P^T   A = 16 dims x 32 keys of V^T (LDS), B = P (registers).
// The A rows are read in a permuted order (key / dim 8 (r / 4) + 4 t + r % 4 for row r of tile t of
// a pair), so that a lane's scores are 8 consecutive keys, the B operand of the P.V product, and
// its outputs runs of 8 dims.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "attn_kernels.h"
#include "clef_hip_attn.h"
#include "split32.h"

namespace clef_hip {
namespace text32 {

constexpr int HD = 256;
constexpr int BLK = 128;                // query rows of a plan block
constexpr int BK = 32;                  // keys per LDS tile
constexpr int NW = 8;                   // waves per workgroup

typedef __attribute__((ext_vector_type(4))) float f32x4;

// Row groups of 16 rows and heads of a full item of `slots` waves, for kv groups of `group` heads: two
// heads where the group is even (a causal item's last tiles are masked for its first rows, so
// fewer rows waste less), one otherwise.
struct Shape {
    int R, k;
};
__host__ __device__ inline Shape f32_shape(int slots, int group) { return group % 2 == 0 ? Shape{slots / 2, 2} : Shape{slots, 1}; }
// Heads of an item that holds only `rows` rows: the largest divisor of the group that fits.
__host__ __device__ inline int f32_heads(int slots, int rows, int group) {
    const int wph = (rows + 15) / 16;
    for (int k = slots / wph; k > 1; k--)
        if (group % k == 0) return k;
    return 1;
}

// Workgroups of a block, for n_blk blocks of T rows in all with `items` items each in `subs` runs of rows, of which the
// last ones hold a short block's rows and the others are empty. Workgroup i goes to shader engine i % 32 (eight XCDs of
// four), busy or not: where the runs with rows fall on the same engines block after block, these take a second
// round while the others idle. A block then gets idle workgroups up to the next count whose multiples bring the
// items of the pass's blocks to all engines alike, at the latest the one that leaves the following block's items where
// its own ended (modulo 32). That is done where
//   the items with rows come unevenly, and the engines hit most get more than their CUs (records x tokens, us:
//   16 / 8 heads, 12 x 64 43.4 -> 29.3; 32 / 4, 200 x 16 541 -> 141; 24 / 4, 200 x 16 164 -> 108), or
//   the items with rows fit the CUs and all workgroups do not (15 / 3, 10 x 45 39.3 -> 25.7; 24 / 4,
//   16 x 64 61.3 -> 37.8), unless they are of one key tile, where idle workgroups cost more (16 x 30 28.3 -> 29.1).
__host__ inline int f32_stride(long n_blk, long T, int items, int subs, long cus) {
    const int layer = items / subs, span = BLK / subs, turn = items & -items, step = turn < 32 ? turn : 32;
    const long rows = n_blk > 0 ? (T + n_blk - 1) / n_blk : 0;   // of a block, rounded up
    const long full = (rows + span - 1) / span * layer;           // its items with rows
    const bool uneven = full % step && n_blk * ((full + step - 1) / step * step) > cus, spill = rows > BK && n_blk * full <= cus && n_blk * items > cus;
    if (!uneven && !spill) return items;
    int stride = items, turns;
    do {
        stride++;
        turns = stride % 32 ? stride & -stride : 32;   // engines that one block's start moves on by at least
    } while ((stride - layer) % 32 && (layer % turns || 32 / turns > n_blk));
    return n_blk * stride < (1L << 32) / (64 * NW) ? stride : items;
}

struct PrepParams {
    const float *qkv;           // [T][row]
    const float *k_norm;        // [256] or NULL
    const int32_t *pos3;
    const float *inv_freq;      // [32]
    const int32_t *kv_tok;      // pass row of each plane row, -1: not written
    float *k_plane, *v_plane;   // [nkv][kvT][256]
    float *rope_cs;             // [T][32][2] or NULL
    int kv_rows, row, nh, nkv, n_rot, kvT;
    float eps;
};

struct Params {
    const float *qkv;
    const float *q_norm;        // [256] or NULL
    const int32_t *pos3;
    const float *inv_freq;
    const float *rope_cs;       // [T][32][2] written by the prep, or NULL
    const float *k_plane, *v_plane;
    const int32_t *blocks;      // the plan's 128-row blocks {q_row0, nq, q_pos0, k_row0, k_len, flag_row, ..}
    void *out;
    int32_t *ovf;
    int row, kvT, nh, nkv, n_rot, causal, gate, out_type;
    int slots;                  // waves of an item that hold rows: 8, or 4 (the others only stage tiles)
    int stride;                 // workgroups of a block: its items, and idle ones behind them (core_f32)
    float eps, scale, f16_lim;
};

// The rotary angle's cos / sin in full FP32 precision (the reference: precise::cos / sin).
__device__ __forceinline__ void rope_cs_f32(const int32_t *pos3, const float *inv_freq, int t, int i, float *c, float *s) {
    const float ang = (float)pos3[3 * (size_t)t + i % 3] * inv_freq[i];
    sincosf(ang, s, c);
}

// K / V prologue, FP32 planes: 32 lanes per (plane row, kv head); lane holds dims lane + 32 j,
// so the rotary pair (i, i + 32), i < 32, sits in one lane. Plane rows with kv_tok -1 are left
// as they are. Head 0's groups also store the rotary cos / sin of their pass row.
__global__ __launch_bounds__(256) void text_prep_kv_f32_kernel(PrepParams p) {
    const long item = (long)blockIdx.x * 8 + (threadIdx.x >> 5);
    const int lane = threadIdx.x & 31;
    if (item >= (long)p.kv_rows * p.nkv) return;
    const int r = (int)(item / p.nkv), kh = (int)(item % p.nkv);
    const int t = p.kv_tok[r];
    if (t < 0) return;
    const float *src = p.qkv + (size_t)t * p.row + (size_t)p.nh * 2 * HD + (size_t)kh * HD;
    float x[8], v[8], ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        x[j] = src[lane + 32 * j];
        v[j] = src[(size_t)p.nkv * HD + lane + 32 * j];
        ss += x[j] * x[j];
    }
    if (p.k_norm) {
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 32);
        const float inv = 1.0f / sqrtf(ss / (float)HD + p.eps);
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = x[j] * inv * p.k_norm[lane + 32 * j];
    }
    if (p.n_rot) {
        float c, s;
        rope_cs_f32(p.pos3, p.inv_freq, t, lane, &c, &s);
        const float x0 = x[0], x1 = x[1];
        x[0] = x0 * c - x1 * s;
        x[1] = x1 * c + x0 * s;
        if (p.rope_cs && kh == 0) *(float2 *)(p.rope_cs + ((size_t)t * 32 + lane) * 2) = make_float2(c, s);
    }
    float *kd = p.k_plane + ((size_t)kh * p.kvT + r) * HD, *vd = p.v_plane + ((size_t)kh * p.kvT + r) * HD;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        kd[lane + 32 * j] = x[j];
        vd[lane + 32 * j] = v[j];
    }
}

// max over the four 16-lane rows of a wave (permlane swaps, VALU only); every lane gets it
__device__ __forceinline__ float xrow_max(float x) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float m = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

// The rows of `rows` (a bit each) of a wave's 16 in plain FP32, for rows whose Q or a key that they see holds an
// infinity, a NaN or a magnitude from 2^55 on (split_bad): FP32 matrix products of operands
// straight from the planes, 16 keys at a time from the record's first, so that a row's bits do not depend on
// the rows beside it. One infinity that all tokens see, 24 / 4 heads: 425 tokens 165 us with the item's first
// run (57 without it; row by row in vector code 2,170), 2,000 tokens 1.0 ms (13.9).
//   S^T = K . Q^T      A = 16 keys x 4 dims, B = Q: lane (g, r16) holds dims 16 c + 4 g + e of row r16.
//   O^T += V^T . P^T   A = dims 64 m + 4 i + e x keys 4 g + v, B = P: O is dims 64 m + 16 g + 4 v + e of row r16.
__device__ __forceinline__ void text_rows_plain(const Params &p, unsigned rows, int q_row0, int q_pos0, int k_row0, int k_len, int h, int kh, int32_t *flag) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const bool mine = (rows >> r16) & 1;
    const int r = mine ? r16 : __builtin_ctz(rows), t = q_row0 + r;
    const float *kbase = p.k_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    const float *vbase = p.v_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    const float *src = p.qkv + (size_t)t * p.row + (size_t)h * 2 * HD;
    f32x4 q[16];
#pragma unroll
    for (int c = 0; c < 16; c++) q[c] = *(const f32x4 *)(src + 16 * c + 4 * g);
    if (p.q_norm) {
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < 16; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) ss += q[c][e] * q[c][e];
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        const float inv = 1.0f / sqrtf(ss / (float)HD + p.eps);
#pragma unroll
        for (int c = 0; c < 16; c++) {
            const f32x4 w = *(const f32x4 *)(p.q_norm + 16 * c + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; e++) q[c][e] = q[c][e] * inv * w[e];
        }
    }
    if (p.n_rot) {
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float cs, sn;
                rope_cs_f32(p.pos3, p.inv_freq, t, 16 * c + 4 * g + e, &cs, &sn);
                const float x0 = q[c][e], x1 = q[c + 2][e];
                q[c][e] = x0 * cs - x1 * sn;
                q[c + 2][e] = x1 * cs + x0 * sn;
            }
    }
    const float sl2 = p.scale * 1.4426950408889634f;
#pragma unroll
    for (int c = 0; c < 16; c++) q[c] *= sl2;
    // keys that the lane's row sees, and the most that one of `rows` does
    const int keys = p.causal ? min(k_len, q_pos0 + r + 1) : k_len;
    const int last = p.causal ? min(k_len, q_pos0 + 32 - __builtin_clz(rows)) : k_len;
    f32x4 o[4][4];
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int e = 0; e < 4; e++) o[m][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (int kb = 0; kb < last; kb += 16) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        // every load goes out before the products (the compiler would wait for each)
        const float *kr = kbase + (size_t)min(kb + r16, k_len - 1) * HD + 4 * g;
        f32x4 k[16], w[2][4];
#pragma unroll
        for (int c = 0; c < 16; c++) k[c] = *(const f32x4 *)(kr + 16 * c);
        auto load_v = [&](int v) {
            const float *vr = vbase + (size_t)min(kb + 4 * g + v, k_len - 1) * HD + 4 * r16;
#pragma unroll
            for (int m = 0; m < 4; m++) w[v & 1][m] = *(const f32x4 *)(vr + 64 * m);
        };
        load_v(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 16; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c][e], q[c][e], s, 0, 0, 0);
        // s[v] is the score (exponent of 2) of key kb + 4g + v for row r16
        float x[4], mx = -INFINITY, rs = 0.f;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            x[v] = kb + 4 * g + v < keys ? s[v] : -INFINITY;
            mx = fmaxf(mx, x[v]);
        }
        const float mn = fmaxf(m_run, xrow_max(mx));
        const float alpha = m_run == -INFINITY ? (mn == -INFINITY ? 1.f : 0.f) : __builtin_amdgcn_exp2f(m_run - mn);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            x[v] = x[v] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x[v] - mn);
            rs += x[v];
        }
        m_run = mn;
        l_run = l_run * alpha + rs;
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[m][e] *= alpha;
        // infinities and NaN of V stay out of the matrix products, whose other rows may not see their keys
        bool special = false;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (v < 3) load_v(v + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float a = w[v & 1][m][e];
                    const bool fin = isfinite(a);
                    special |= !fin;
                    o[m][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(fin ? a : 0.f, x[v], o[m][e], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
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
                const float *vr = vbase + (size_t)min(kb + j, k_len - 1) * HD + 16 * g;
#pragma unroll
                for (int m = 0; m < 4; m++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const f32x4 a = *(const f32x4 *)(vr + 64 * m + 4 * v);
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (!isfinite(a[e]) && kb + j < keys) o[m][e][v] = fmaf(pj, a[e], o[m][e][v]);
                    }
            }
        }
    }
    float l_row = l_run;
    l_row += __shfl_xor(l_row, 16);
    l_row += __shfl_xor(l_row, 32);
    if (!mine) return;
    const float il = l_row > 0.f ? 1.0f / l_row : 0.f;
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int d = 64 * m + 16 * g + 4 * v;
            f32x4 w;
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = o[m][e][v] * il;
            if (p.gate) {
                const f32x4 gv = *(const f32x4 *)(src + HD + d);
#pragma unroll
                for (int e = 0; e < 4; e++) w[e] = w[e] * sigmoidf(gv[e]);
            }
            store_out4(p.out, (size_t)t * p.nh * HD + (size_t)h * HD + d, w, p.out_type, p.f16_lim, flag);
        }
}

// Work items are (block, R x 16 rows of it, k heads of a kv group, kv head), the plan's longest-first
// blocks outermost, each block's last rows first, kv heads innermost (an XCD then streams the K / V
// of few of them), one workgroup each. An item of few rows runs more heads (f32_heads), and the
// items of the heads it took are empty, as are those past a block's rows.
//
// Per 32-key tile: barrier; S(t) while V(t) is split into LDS; barrier; softmax; P.V(t) while
// K(t + 1) is split. The operand staged beside a product is the one the product does not read, so
// one buffer each is enough; its loads go out a phase ahead into registers that K and V share.
__global__ __launch_bounds__(64 * NW) void attn_text_f32_kernel(Params p) {
    constexpr int PL = BK * HD * 2, KV = 3 * PL;           // bytes of one bf16 plane; the V^T planes
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * KV];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int group = p.nh / p.nkv;
    const Shape shape = f32_shape(p.slots, group);
    const int span = 16 * shape.R, n_sub = BLK / span, n_ch = group / shape.k;
    const split32::Weights wt;
    // per-lane LDS byte addresses of the operand reads (plane h)
    const unsigned lds0 = split32::lds_offset(smem);
    unsigned ka[4];   // 32-dim step c, c % 4: K row of S^T A row r16 in subtile 0 (+ 256 c / 4; subtile 1: + 4 rows)
#pragma unroll
    for (int c = 0; c < 4; c++) ka[c] = lds0 + (8 * (r16 >> 2) + (r16 & 3)) * (2 * HD) + (((4 * c + g) ^ r16) * 16);
    unsigned va[2];   // V^T row of O^T A row r16 in dim tiles 0 and 1 (tiles 2u + w: + 32 u rows)
#pragma unroll
    for (int w = 0; w < 2; w++)
        va[w] = lds0 + KV + (8 * (r16 >> 2) + 4 * w + (r16 & 3)) * (2 * BK) + ((g ^ (-(r16 >> 2) & 3) ^ w) * 16);

    const int bi = blockIdx.x / p.stride, item = blockIdx.x - bi * p.stride;
    const int kh = item % p.nkv, ic = item / p.nkv % n_ch, sub = item / p.nkv / n_ch;
    const int32_t *blk = p.blocks + 8 * bi;
    const int r0 = span * (n_sub - 1 - sub), rows = min(span, blk[1] - r0);
    if (sub >= n_sub || rows <= 0) return;
    const int kk = f32_heads(p.slots, rows, group), wph = (rows + 15) / 16;
    if (ic * kk >= group) return;
    const int slot = wave / wph;
    const bool live = slot < kk;
    const int h = kh * group + ic * kk + (live ? slot : 0);
    const int q_row0 = blk[0] + r0 + (live ? 16 * (wave - slot * wph) : 0), q_pos0 = blk[2] + q_row0 - blk[0];
    const int nq = live ? min(16, blk[0] + r0 + rows - q_row0) : 0;
    const int k_row0 = blk[3], k_len = p.causal ? min(blk[4], blk[2] + r0 + rows) : blk[4];
    const int whole = p.causal ? min(k_len, blk[2] + r0 + 1) : k_len;   // keys that every row of the item sees
    int32_t *const flag = p.ovf ? p.ovf + blk[5] : nullptr;
    const int n_tiles = (k_len + BK - 1) / BK;
    // keys this wave's rows see, and the tiles it runs
    const int my_len = live ? (p.causal ? min(k_len, q_pos0 + nq) : k_len) : 0;
    const bool q_valid = r16 < nq;
    const float *const kbase = p.k_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    const float *const vbase = p.v_plane + ((size_t)kh * p.kvT + k_row0) * HD;
    float amax = 0.f;

    // ---- tile staging, two pieces a thread. Piece e: K dims 8 c .. 8 c + 7
    // of one key, V keys 8 kg .. 8 kg + 7 of one dim; each load is a uniform base plus a
    // 32-bit lane offset. Keys past the item's range become zeros: their zero probabilities
    // then give zero products, and what lies there cannot flag the item. So do values of V that
    // are left to plain arithmetic, in tiles that some row sees in part.
    float raw[2][8];
    const unsigned ko = 32u * tid, vo = (tid >> 8) * (8u * HD * 4u) + (tid & 255) * 4u;
    auto load_k = [&](int kb) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const char *s = (const char *)(kbase + (size_t)(kb + 2 * NW * e) * HD);
            const f32x4 a = *(const f32x4 *)(s + ko), b = *(const f32x4 *)(s + ko + 16);
#pragma unroll
            for (int j = 0; j < 4; j++) { raw[e][j] = a[j]; raw[e][4 + j] = b[j]; }
        }
    };
    auto load_v = [&](int kb) {
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const char *s = (const char *)(vbase + (size_t)(kb + 2 * NW * e + j) * HD);
                raw[e][j] = *(const float *)(s + vo);
            }
    };
    // K chunk c of key 8a + 4t + b sits at position c ^ (4a + b), V^T chunk kg of dim d at
    // kg ^ (-(d / 8) % 4) ^ ((d / 4) % 2): the lanes one step of a read or write serves hit
    // distinct 16-byte slots.
    const unsigned dk = (tid >> 5) * (2 * HD) + (((tid & 31) ^ (((tid >> 5) & 3) | (((tid >> 5) >> 3) << 2))) * 16);
    const unsigned dv = KV + (tid & 255) * (2 * BK) + (((tid >> 8) ^ (-((tid & 255) >> 3) & 3) ^ ((tid >> 2) & 1)) * 16);
    // piece e lies 2 NW e keys on, or NW e / 4 chunks: no carry into the bits of the thread's own
    auto dst_k = [&](int e) { return smem + (dk ^ (unsigned)(((2 * NW * e) >> 3 << 2) * 16)) + 2 * NW * e * (2 * HD); };
    auto dst_v = [&](int e) { return smem + (dv ^ (unsigned)((NW / 4 * e) * 16)); };
    auto put = [&](auto DST, auto V) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            amax = split32::split_amax(amax, raw[e]);
            if constexpr (decltype(V)::value) split32::scale_v(raw[e]);
            const split32::Parts x = split32::split8(raw[e], wt);
            uint8_t *const dst = DST(e);
            *(bf16x8 *)dst = x.h;
            *(bf16x8 *)(dst + PL) = x.m;
            *(bf16x8 *)(dst + 2 * PL) = x.l;
        }
    };
    auto put_k = [&](int kb) {
        if (kb + BK > k_len) {
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int j = 0; j < 8; j++) raw[e][j] = kb + (tid >> 5) + 2 * NW * e < k_len ? raw[e][j] : 0.f;
        }
        put(dst_k, std::false_type{});
    };
    auto put_v = [&](int kb) {
        if (kb + BK > whole) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
#pragma unroll
                for (int j = 0; j < 8; j++) raw[e][j] = kb + 8 * (tid >> 8) + 2 * NW * e + j < k_len ? raw[e][j] : 0.f;
                amax = split32::split_amax(amax, raw[e]);
#pragma unroll
                for (int j = 0; j < 8; j++) raw[e][j] = split32::split_bad(raw[e][j]) ? 0.f : raw[e][j];
            }
        }
        put(dst_v, std::true_type{});
    };

    load_k(0);
    // ---- Q prologue: lane holds Q[row r16][32 c + 8 g + j], the B operand of step c:
    // normalised, rotated (pair i < 32 is chunks 0 and 1 of the lane) and scaled by
    // scale * log2 e (the scores then are exponents of 2), in FP32, then split
    bf16x8 qh[8], qm[8], ql[8];
    {
        // every load goes out before the first is used
        const int t = q_row0 + (q_valid ? r16 : 0);
        const float *qs = p.qkv + (size_t)t * p.row + (size_t)h * 2 * HD + 8 * g;
        float x[8][8];
        f32x4 w[8][2], cs[4];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const f32x4 a = *(const f32x4 *)(qs + 32 * c), b = *(const f32x4 *)(qs + 32 * c + 4);
#pragma unroll
            for (int j = 0; j < 4; j++) { x[c][j] = a[j]; x[c][4 + j] = b[j]; }
        }
        // without norms or a table, the pass's own rows stand in (loaded, not used)
        const float *ws = p.q_norm ? p.q_norm + 8 * g : qs, *ts = p.rope_cs ? p.rope_cs + (size_t)t * 64 + 16 * g : qs;
#pragma unroll
        for (int c = 0; c < 8; c++)
#pragma unroll
            for (int i = 0; i < 2; i++) w[c][i] = *(const f32x4 *)(ws + 32 * c + 4 * i);
#pragma unroll
        for (int q = 0; q < 4; q++) cs[q] = *(const f32x4 *)(ts + 4 * q);   // cos, sin of pairs 8g + 2q, 8g + 2q + 1
        if (p.n_rot && !p.rope_cs) {
            // no table: the wave evaluates its rows' angles into LDS (the V^T region is free)
            float2 *tab = (float2 *)(smem + KV) + 16 * 32 * wave;
            for (int i = lane; i < 16 * 32; i += 64) {
                const int row = i >> 5;
                float c, s;
                rope_cs_f32(p.pos3, p.inv_freq, q_row0 + (row < nq ? row : 0), i & 31, &c, &s);
                tab[i] = make_float2(c, s);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) cs[q] = *(const f32x4 *)(tab + 32 * r16 + 8 * g + 2 * q);
        }
        if (p.q_norm) {
            float ss = 0.f;
#pragma unroll
            for (int c = 0; c < 8; c++)
#pragma unroll
                for (int j = 0; j < 8; j++) ss += x[c][j] * x[c][j];
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            const float inv = 1.0f / sqrtf(ss / (float)HD + p.eps);
#pragma unroll
            for (int c = 0; c < 8; c++)
#pragma unroll
                for (int j = 0; j < 8; j++) x[c][j] = x[c][j] * inv * w[c][j >> 2][j & 3];
        }
        if (p.n_rot) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float c = cs[j >> 1][2 * (j & 1)], s = cs[j >> 1][2 * (j & 1) + 1];
                const float x0 = x[0][j], x1 = x[1][j];
                x[0][j] = x0 * c - x1 * s;
                x[1][j] = x1 * c + x0 * s;
            }
        }
        const float sl2 = p.scale * 1.4426950408889634f;
#pragma unroll
        for (int c = 0; c < 8; c++) {
#pragma unroll
            for (int j = 0; j < 8; j++) x[c][j] *= sl2;
            amax = split32::split_amax(amax, x[c]);
            const split32::Parts s = split32::split8(x[c], wt);
            qh[c] = s.h; qm[c] = s.m; ql[c] = s.l;
        }
    }
    put_k(0);
    load_v(0);

    f32x4 o[16];
#pragma unroll
    for (int n = 0; n < 16; n++) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the running maximum starts at the lowest finite value: a row that has seen no key yet
    // then needs no case of its own
    float m_run = -3.4028235e38f, l_run = 0.f;
    // every LDS access of the phase is done; the loads in flight stay so
    auto phase_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int t = 0; t < n_tiles; t++) {
        const int kb = t * BK;
        const bool mine = kb < my_len;   // wave-uniform
        phase_barrier();                 // K(t) is in place; V(t - 1) has been read
        // S^T: two 16-key subtiles, eight 32-dim steps; the hh terms in one accumulator, the
        // smaller ones in another
        split32::Ring ring;
        f32x4 s[2], sx[2];
#pragma unroll
        for (int u = 0; u < 2; u++) s[u] = sx[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (mine) split32::ring_start<PL, 0, 4 * 2 * HD>(ring, ka[0], ka[0]);
        const bool more = t + 1 < n_tiles;
        put_v(kb);
        if (more) {
            load_k(kb + BK);
        } else {   // nothing: but a value that seemed to live on would be copied before its split
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int j = 0; j < 8; j++) asm volatile("" : "=v"(raw[e][j]));
        }
        if (mine) {
            split32::sfor<8>([&](auto I) {
                constexpr int i = decltype(I)::value, n = i + 1, o8 = 256 * (n / 4);
                split32::ring_step<PL, (n < 8), o8, o8 + 4 * 2 * HD>(ring, ka[n % 4], ka[n % 4], s[0], s[1], sx[0], sx[1], qh[i], qm[i], ql[i]);
            });
        }
        phase_barrier();                 // V(t) is in place; K(t) has been read
        if (mine) split32::ring_start<PL, 0, 0>(ring, va[0], va[1]);
        if (more) {
            put_k(kb + BK);
            load_v(kb + BK);
        }
        if (mine) {
            // x[4 u + v] is the score (exponent of 2) of key kb + 8g + 4u + v for row r16
            float x[8], mx, rs = 0.f;
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = s[j >> 2][j & 3] + sx[j >> 2][j & 3];
            if (kb + BK > k_len || (p.causal && kb + BK - 1 > q_pos0)) {
                const int lim = (p.causal ? min(k_len - 1, q_pos0 + r16) : k_len - 1) - kb - 8 * g;
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = j <= lim ? x[j] : -INFINITY;
            }
            mx = x[0];
#pragma unroll
            for (int j = 1; j < 8; j++) mx = fmaxf(mx, x[j]);
            const float mn = fmaxf(m_run, xrow_max(mx));
            const float alpha = __builtin_amdgcn_exp2f(m_run - mn);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                x[j] = split32::P_SCALE * __builtin_amdgcn_exp2f(x[j] - mn);   // a masked key's -inf gives 0
                rs += x[j];
            }
            m_run = mn;
            l_run = l_run * alpha + rs;
            if (__any(alpha != 1.f)) {   // in place (as plain C++ the other path copies the registers)
#pragma unroll
                for (int n = 0; n < 16; n++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        float d = o[n][v];
                        asm("v_mul_f32 %0, %1, %0" : "+v"(d) : "v"(alpha));
                        o[n][v] = d;
                    }
            }
            const split32::Parts pp = split32::split8(x, wt);
            // O^T += V^T . P^T: pairs of 16-dim tiles, the six terms smallest first
            split32::sfor<8>([&](auto I) {
                constexpr int i = decltype(I)::value, o8 = 32 * (i + 1) * 2 * BK;
                split32::ring_step<PL, (i + 1 < 8), o8, o8>(ring, va[0], va[1], o[2 * i], o[2 * i + 1], o[2 * i], o[2 * i + 1], pp.h, pp.m, pp.l);
            });
        }
    }

    // ---- epilogue: O = O^T / l, times sigmoid(gate). Tiles 2u, 2u + 1 of lane (g, r16) are
    // dims 32 u + 8 g .. + 7 of row r16.
    float l_row = l_run;
    l_row += __shfl_xor(l_row, 16);
    l_row += __shfl_xor(l_row, 32);
    bool plain = false;
    if (__syncthreads_or(!split32::split_fine(amax))) {   // also: the tiles' last reads are done
        const int first = split32::first_bad_key<HD>(kbase, vbase, k_len, (int *)smem);
        int own = 0;
#pragma unroll
        for (int c = 0; c < 8; c++) own |= split32::query_bad(qh[c]);
        own |= __shfl_xor(own, 16);
        own |= __shfl_xor(own, 32);
        plain = q_valid && (own || first < (p.causal ? q_pos0 + r16 + 1 : k_len));
    }
    if (q_valid && !plain) {
        const float il = l_row > 0.f ? (1.0f / split32::V_SCALE) / l_row : 0.f;
        const size_t t = (size_t)(q_row0 + r16);
        const size_t obase = t * p.nh * HD + (size_t)h * HD + 8 * g;
        if (p.gate) {   // every gate load goes out before the first store
            const float *grow = p.qkv + t * p.row + (size_t)h * 2 * HD + HD + 8 * g;
            f32x4 gv[16];
#pragma unroll
            for (int n = 0; n < 16; n++) gv[n] = *(const f32x4 *)(grow + 32 * (n >> 1) + 4 * (n & 1));
#pragma unroll
            for (int n = 0; n < 16; n++)
#pragma unroll
                for (int v = 0; v < 4; v++) o[n][v] = o[n][v] * il * sigmoidf(gv[n][v]);
        } else {
#pragma unroll
            for (int n = 0; n < 16; n++) o[n] *= il;
        }
        auto store = [&](const int type) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                float w[8];
#pragma unroll
                for (int j = 0; j < 8; j++) w[j] = o[2 * u + (j >> 2)][j & 3];
                store_out8(p.out, obase + 32 * u, w, type, p.f16_lim, flag);
            }
        };
        if (p.out_type == CLEF_HIP_OUT_F32) store(CLEF_HIP_OUT_F32);
        else if (p.out_type == CLEF_HIP_OUT_BF16) store(CLEF_HIP_OUT_BF16);
        else store(CLEF_HIP_OUT_F16);
    }
    const unsigned plain_rows = (unsigned)__ballot(plain) & 0xffffu;
    if (plain_rows) text_rows_plain(p, plain_rows, q_row0, q_pos0, k_row0, k_len, h, kh, flag);
}

}  // namespace text32
}  // namespace clef_hip
