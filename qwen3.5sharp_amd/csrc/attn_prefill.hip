// Gated GQA attention prefill for T tokens of one sequence starting at row
// `start` of its KV cache.
//
// Reference: Qwen35Model.PrefillAttention after the projections
// (src/Qwen35Sharp.Model/Qwen35Model.Prefill.cs:113-149): q|gate
// de-interleave, K/V written into cache rows start.., NeoX RoPE then (1+w)
// RMSNorm on q and on the cached K rows, causal softmax attention over
// start+T rows with scale 1/sqrt(head_dim), times sigmoid(gate).
//
// Two forms.  attn_split_* (below) is the one that runs; the fp32 form takes
// calls without room for its workspace and values outside its range:
//
//  1. attn_prefill_prep: rotate/norm K into the cache, copy V into the cache.
//  2. attn_prefill_flash: causal flash attention on fp32 MFMA, one workgroup
//     per (group of up to 4 q heads sharing a kv head, 16-row query block),
//     which rotates and norms its q rows (scale folded in) in registers,
//     its key range split between two halves of the workgroup, K/V streamed
//     through LDS in 32-row tiles, online softmax; the [T][kvLen] score
//     matrix is never materialised.
#include <algorithm>
#include <array>
#include <type_traits>

#include "common.h"
#include "q35mix_internal.h"

namespace q35 {
namespace {

// 1 / (1 + e^-x) to fp32 precision in a dozen instructions: the exponential
// with the rounding error of its base-2 argument made good, the reciprocal
// with one Newton step (expf and a division are 45).
__device__ __forceinline__ float sigmoid_full(float x) {
    const float n = __builtin_amdgcn_fmed3f(-x, -88.0f, 88.0f);    // (past it 0 and 1 in any case)
    const float l2 = 1.44269502e+0f, l2lo = 1.92596303e-8f, ln2 = 0.693147182f;   // log2(e) as a sum, ln 2
    const float t = n * l2, d = fmaf(n, l2lo, fmaf(n, l2, -t));
    const float p = __builtin_amdgcn_exp2f(t), s = 1.0f + fmaf(p * ln2, d, p);
    const float r = __builtin_amdgcn_rcpf(s);
    return x != x ? x : fmaf(fmaf(-s, r, 1.0f), r, r);
}

__global__ __launch_bounds__(kWave) void attn_prefill_prep(
    const float* __restrict__ knew, const float* __restrict__ vnew, const float* __restrict__ k_norm,
    float* __restrict__ K, float* __restrict__ V, const float* __restrict__ rope_cos,
    const float* __restrict__ rope_sin, int start, int nkv, int cap, float eps) {
    const int t = blockIdx.x, kvh = blockIdx.y, lane = threadIdx.x;
    const int pos = start + t;
    const int kv_dim = nkv * kHd;
    float4 x = *reinterpret_cast<const float4*>(knew + (size_t)t * kv_dim + kvh * kHd + 4 * lane);
    x = rope_norm_row(x, lane, rope_cos + (size_t)pos * kRopeHalf, rope_sin + (size_t)pos * kRopeHalf, k_norm, eps, 1.0f);
    // Head-major cache: row pos of kv head kvh at (kvh * cap + pos) * 256.
    const size_t row = ((size_t)kvh * cap + pos) * kHd;
    *reinterpret_cast<float4*>(K + row + 4 * lane) = x;
    const float4 v = *reinterpret_cast<const float4*>(vnew + (size_t)t * kv_dim + kvh * kHd + 4 * lane);
    *reinterpret_cast<float4*>(V + row + 4 * lane) = v;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int QR = 16;          // query rows per workgroup (per head)
constexpr int KT = 32;          // key rows per tile
constexpr int LDKV = kHd + 4;   // padded LDS row stride of the K tiles
constexpr int LDVT = KT + 4;    // padded LDS row stride of the transposed V tiles

// Causal flash attention on fp32 MFMA (v_mfma_f32_16x16x4f32).  Workgroup =
// (head group y, 16 query rows) in two halves of 4 waves: half 0 takes the
// first ceil(n/2) of the block's n key tiles, half 1 the rest, each with its
// own K/V tiles in LDS, and half 0 merges the two online-softmax states at
// the end (max, sum and the unnormalised output rescaled to the common max).
// So every workgroup keeps 8 waves busy on half of its block's key range, and
// one workgroup a CU, dispatched heaviest first, balances the causal work
// over the CUs.  Within a half the group is hg = min(4, q heads per kv head)
// q heads hg y .. hg y + hg - 1 of one kv head, and wave w of the half is q
// head hg y + w, so the group's q heads share every K/V tile (with fewer than
// 4 heads the spare waves repeat the last head and store nothing).  Per
// 32-row key tile a wave computes S^T = K Q^T (positions x queries), so each
// lane's D column is one query: the online-softmax max/sum and the rescale of
// O^T = V^T P^T are per lane, and S^T's D tile feeds P^T = B operand register
// by register.  Lane l = 16g + c: Q operand holds Q[row c][64g + s], s < 64
// (reduction index of instruction s for lane group g), O^T register r of
// block db holds O[row c][16 db + 4g + r].  V tiles are stored transposed
// (dims x positions), so a lane's four P.V operands of a 16-position block are
// one 16-byte read; P.V runs four output blocks at a time (four independent
// accumulation chains, each in the order pb, s2), S one key-row block ahead
// in its operand reads.  The next K tile goes to LDS by buffer loads straight
// into LDS once every wave is past S, the next V tile into registers.
// K tiles (row-major) and V tiles (transposed: dims x positions, so a
// lane's P.V operands for 4 positions are one 16-byte read) of each half;
// at the end, the merge's exchange area.
struct Tiles {
    float k[KT][LDKV];
    float vt[kHd][LDVT];
};

// What a q row needs besides its values.
struct QRows {
    const float *q_gate, *q_norm, *rope_cos, *rope_sin;
    float eps;
};

// Query block qb (16 subs rows) of head group y; every thread of the
// workgroup's 8 waves.  With subs > 1 the spare waves take further 16 rows.
// KEYS false: the halves take a block each, 2 qb and 2 qb + 1, and all its keys.
template <bool KEYS>
__device__ __forceinline__ void flash_fp32_block(
    Tiles* smem, const QRows& Q, const float* __restrict__ K, const float* __restrict__ V,
    float* __restrict__ out, int start, int T, int nh, int nkv, int hg, int cap, int qb, int y, int subs) {
    const float* q_gate = Q.q_gate;
    const int kvh = y * hg / (nh / nkv);
    const int tid = threadIdx.x, lane = tid & 63;
    // Wave-uniform (readfirstlane): the K tile loads take them as scalar
    // offsets and LDS bases.
    const int half = __builtin_amdgcn_readfirstlane(tid >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, htid = tid & 255;
    const int g = lane >> 4, c16 = lane & 15;
    const bool stores = wave < hg * subs;    // uniform per wave
    const int unit = min(wave, hg * subs - 1), h = hg * y + unit % hg;
    const int r0 = ((KEYS ? qb : 2 * qb + half) * subs + unit / hg) * QR;
    const int blk_len = start + min(T - 1, (qb + 1) * (KEYS ? 1 : 2) * subs * QR - 1) + 1;
    const int my_t = min(r0 + c16, T - 1);
    const int my_len = start + my_t + 1;
    // Key tiles of this half: [t_begin, t_begin + n_iter), the last one past
    // blk_len (fully masked) when half 1 has one tile fewer.
    const int n_tiles = (blk_len + KT - 1) / KT, n_iter = KEYS ? (n_tiles + 1) / 2 : n_tiles;
    const int p_begin = KEYS ? half * n_iter * KT : 0;
    // Head-major cache: kv head kvh's rows are [cap][256] from kvh * cap * 256.
    const float* Kh = K + (size_t)kvh * cap * kHd;
    const float* Vh = V + (size_t)kvh * cap * kHd;

    float (*Ks)[LDKV] = smem[half].k;
    float (*Vt)[LDVT] = smem[half].vt;

    // q row c16, dims 64 g + s: RoPE over the pairs (d, d + 32) of lanes g = 0,
    // then the (1 + w) norm with the attention scale (rope_norm_row's steps).
    float qreg[64];
    {
        const float* qrow = q_gate + ((size_t)my_t * nh + h) * 2 * kHd + 64 * g;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const float4 x = *reinterpret_cast<const float4*>(qrow + 4 * u);
            qreg[4 * u] = x.x; qreg[4 * u + 1] = x.y; qreg[4 * u + 2] = x.z; qreg[4 * u + 3] = x.w;
        }
        const float* cs = Q.rope_cos + (size_t)(my_len - 1) * kRopeHalf;
        const float* sn = Q.rope_sin + (size_t)(my_len - 1) * kRopeHalf;
        if (g == 0)
#pragma unroll
            for (int s = 0; s < 32; ++s) {
                const float x0 = qreg[s], x1 = qreg[s + 32];
                qreg[s] = x0 * cs[s] - x1 * sn[s];
                qreg[s + 32] = x0 * sn[s] + x1 * cs[s];
            }
        float ss = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            float p = 0.0f;
#pragma unroll
            for (int s = 0; s < 8; ++s) p += qreg[8 * u + s] * qreg[8 * u + s];
            ss += p;
        }
        ss = xor16_sum(ss);
        ss = xor32_sum(ss);
        const float scale = 1.0f / sqrtf(ss / 256.0f + Q.eps), post = 1.0f / sqrtf((float)kHd);
#pragma unroll
        for (int s = 0; s < 64; ++s) qreg[s] = qreg[s] * scale * (1.0f + Q.q_norm[64 * g + s]) * post;
    }
    f32x4 O[16];
#pragma unroll
    for (int db = 0; db < 16; ++db) O[db] = {0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.0f;

    // Staging.  K: wave w of the half loads rows w, w + 4, ... of the tile
    // by buffer loads straight into LDS (one 1 KiB row a load).  V (stored
    // transposed): thread row htid % 32, float4 columns htid / 32 + 8 i, so
    // that the transposed stores of 32 lanes land on 32 consecutive words.
    // Rows past blk_len read row 0 instead (finite data; their scores are
    // masked), so no select waits on the loads, and the refill is
    // unconditional.
    // The host keeps start + T <= kPrefillMaxRows = 2^21 rows, so a row's
    // offset fits 31 bits and its last 16-byte load ends at most at byte 2^31:
    // the range is whole rows, up to exactly 2^31 bytes (the 32-bit
    // num_records field is unsigned; 0x80000000 as its bit pattern).
    const uint32_t krange = (uint32_t)(std::min<size_t>((size_t)cap, (size_t)kPrefillMaxRows) * kHd * sizeof(float));
    const __amdgpu_buffer_rsrc_t krs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Kh), 0, (int)krange, 0x00020000);
    auto load_k = [&](int p0) {
#pragma unroll
        for (int i = 0; i < KT / 4; ++i) {
            const int r = wave + 4 * i, p = p0 + r;
            dma_b128(krs, &Ks[r][0], 16u * lane, (uint32_t)(p < blk_len ? p : 0) * kHd * sizeof(float));
        }
    };
    const int vrow = htid & 31, vc4 = htid >> 5;
    float4 sv0, sv1, sv2, sv3, sv4, sv5, sv6, sv7;
#define Q35_LOAD_ROW(i, p0)                                                                  \
    {                                                                                      \
        const int pv = (p0) + vrow;                                                        \
        sv##i = *reinterpret_cast<const float4*>(Vh + (size_t)(pv < blk_len ? pv : 0) * kHd +  \
                                                 4 * (vc4 + 8 * (i)));                      \
    }
#define Q35_LOAD_TILE(p0)                                                                    \
    Q35_LOAD_ROW(0, p0) Q35_LOAD_ROW(1, p0) Q35_LOAD_ROW(2, p0) Q35_LOAD_ROW(3, p0)            \
    Q35_LOAD_ROW(4, p0) Q35_LOAD_ROW(5, p0) Q35_LOAD_ROW(6, p0) Q35_LOAD_ROW(7, p0)
#define Q35_STORE_ROW(i)                                                                     \
    Vt[4 * (vc4 + 8 * (i)) + 0][vrow] = sv##i.x;                                            \
    Vt[4 * (vc4 + 8 * (i)) + 1][vrow] = sv##i.y;                                            \
    Vt[4 * (vc4 + 8 * (i)) + 2][vrow] = sv##i.z;                                            \
    Vt[4 * (vc4 + 8 * (i)) + 3][vrow] = sv##i.w;
    load_k(p_begin);
    Q35_LOAD_TILE(p_begin)
    for (int it = 0; it < n_iter; ++it) {
        const int p0 = p_begin + it * KT;
        // The K tile has landed and every wave is past the previous P.V.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        Q35_STORE_ROW(0) Q35_STORE_ROW(1) Q35_STORE_ROW(2) Q35_STORE_ROW(3)
        Q35_STORE_ROW(4) Q35_STORE_ROW(5) Q35_STORE_ROW(6) Q35_STORE_ROW(7)
        __builtin_amdgcn_sched_barrier(0);

        // S^T for positions p0 + 16 pb + (4g + r), queries c16.
        f32x4 st[2];
        {
            f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
            float4 a0 = *reinterpret_cast<const float4*>(&Ks[c16][64 * g]);
            float4 a1 = *reinterpret_cast<const float4*>(&Ks[16 + c16][64 * g]);
            auto products = [&](int u) {
                acc0 = mfma16(a0.x, qreg[4 * u], acc0);
                acc1 = mfma16(a1.x, qreg[4 * u], acc1);
                acc0 = mfma16(a0.y, qreg[4 * u + 1], acc0);
                acc1 = mfma16(a1.y, qreg[4 * u + 1], acc1);
                acc0 = mfma16(a0.z, qreg[4 * u + 2], acc0);
                acc1 = mfma16(a1.z, qreg[4 * u + 2], acc1);
                acc0 = mfma16(a0.w, qreg[4 * u + 3], acc0);
                acc1 = mfma16(a1.w, qreg[4 * u + 3], acc1);
            };
#pragma unroll
            for (int u = 0; u < 15; ++u) {
                const float4 n0 = *reinterpret_cast<const float4*>(&Ks[c16][64 * g + 4 * (u + 1)]);
                const float4 n1 = *reinterpret_cast<const float4*>(&Ks[16 + c16][64 * g + 4 * (u + 1)]);
                products(u);
                a0 = n0; a1 = n1;
            }
            // Every wave has its last operands (the K tile is free) and the V
            // tile is stored: refill K, load the next V into registers.  The
            // last products run behind the barrier.
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (it + 1 < n_iter) {
                load_k(p0 + KT);
                Q35_LOAD_TILE(p0 + KT)
            }
            products(15);
            st[0] = acc0; st[1] = acc1;
        }
#undef Q35_LOAD_ROW
#undef Q35_LOAD_TILE
#undef Q35_STORE_ROW
        // Online softmax down this lane's query column.  A column with no
        // unmasked position yet (half 1 only) keeps m = -inf, l = 0, O = 0.
        float mt = m_run;
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = p0 + 16 * pb + 4 * g + r;
                if (p >= my_len) st[pb][r] = -INFINITY;
                mt = fmaxf(mt, st[pb][r]);
            }
        mt = xor16_max(mt);
        mt = xor32_max(mt);
        const bool live = mt != -INFINITY;
        const float alpha = live ? __expf(m_run - mt) : 1.0f;
        float ls = 0.0f;
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = live ? __expf(st[pb][r] - mt) : 0.0f;
                st[pb][r] = e;
                ls += e;
            }
        ls = xor16_sum(ls);
        ls = xor32_sum(ls);
        l_run = l_run * alpha + ls;
        m_run = mt;
        // O^T = alpha O^T + V^T P^T.
#pragma unroll
        for (int db = 0; db < 16; ++db) O[db] = O[db] * alpha;
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int dq = 0; dq < 4; ++dq) {
                float4 v[4];
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    v[d] = *reinterpret_cast<const float4*>(&Vt[16 * (4 * dq + d) + c16][16 * pb + 4 * g]);
#pragma unroll
                for (int d = 0; d < 4; ++d) O[4 * dq + d] = mfma16(v[d].x, st[pb][0], O[4 * dq + d]);
#pragma unroll
                for (int d = 0; d < 4; ++d) O[4 * dq + d] = mfma16(v[d].y, st[pb][1], O[4 * dq + d]);
#pragma unroll
                for (int d = 0; d < 4; ++d) O[4 * dq + d] = mfma16(v[d].z, st[pb][2], O[4 * dq + d]);
#pragma unroll
                for (int d = 0; d < 4; ++d) O[4 * dq + d] = mfma16(v[d].w, st[pb][3], O[4 * dq + d]);
            }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    float inv;
    if constexpr (KEYS) {
        // Merge: half 1 hands (m, l, O) to half 0 through LDS (the tile
        // buffers, free after the last barrier of the loop).
        static_assert(4 * 64 * 66 * sizeof(float) <= sizeof(Tiles), "merge exchange fits one half's tiles");
        float* xch = &smem[0].k[0][0];
        float* xo = xch + (size_t)(wave * 64 + lane) * 64;
        float* xml = xch + (size_t)4 * 64 * 64 + (size_t)(wave * 64 + lane) * 2;
        __syncthreads();
        if (half == 1) {
#pragma unroll
            for (int db = 0; db < 16; ++db)
                *reinterpret_cast<float4*>(xo + 4 * db) = make_float4(O[db][0], O[db][1], O[db][2], O[db][3]);
            xml[0] = m_run;
            xml[1] = l_run;
        }
        __syncthreads();
        if (half == 1) return;
        const float m1 = xml[0], l1 = xml[1];
        const float m = fmaxf(m_run, m1);
        const float a0 = __expf(m_run - m), a1 = m1 == -INFINITY ? 0.0f : __expf(m1 - m);
        inv = 1.0f / (l_run * a0 + l1 * a1);
#pragma unroll
        for (int db = 0; db < 16; ++db) {
            const float4 o1 = *reinterpret_cast<const float4*>(xo + 4 * db);
            O[db][0] = O[db][0] * a0 + o1.x * a1;
            O[db][1] = O[db][1] * a0 + o1.y * a1;
            O[db][2] = O[db][2] * a0 + o1.z * a1;
            O[db][3] = O[db][3] * a0 + o1.w * a1;
        }
    } else {
        inv = 1.0f / l_run;
    }
    const int t = r0 + c16;
    if (t >= T || !stores) return;
    const float* grow = q_gate + ((size_t)t * nh + h) * 2 * kHd + kHd;
    float* orow = out + ((size_t)t * nh + h) * kHd;
#pragma unroll
    for (int db = 0; db < 16; ++db) {
        const int d0 = 16 * db + 4 * g;
        const float4 gt = *reinterpret_cast<const float4*>(grow + d0);
        float4 r;
        r.x = O[db][0] * inv * sigmoid_full(gt.x);
        r.y = O[db][1] * inv * sigmoid_full(gt.y);
        r.z = O[db][2] * inv * sigmoid_full(gt.z);
        r.w = O[db][3] * inv * sigmoid_full(gt.w);
        *reinterpret_cast<float4*>(orow + d0) = r;
    }
}

__global__ __launch_bounds__(512, 1) void attn_prefill_flash(
    QRows Q, const float* __restrict__ K, const float* __restrict__ V, float* __restrict__ out, int start, int T, int nh,
    int nkv, int hg, int cap) {
    __shared__ Tiles smem[2];
    const int groups = nh / hg, nqb = (T + QR - 1) / QR;
    const int rank = blockIdx.x;                 // heaviest query blocks first
    flash_fp32_block<true>(smem, Q, K, V, out, start, T, nh, nkv, hg, cap, nqb - 1 - rank / groups, rank % groups, 1);
}

// ---------------------------------------------------------------- split fp16

// The same attention on v_mfma_f32_16x16x32_f16: every fp32 operand is the sum
// of two fp16 values (11 + 11 bits and the second one's sign: relative error at
// most 2^-23) after a power-of-two scale that puts the largest of its tile
// (K, V), row (Q) or range (P) at 2^13 .. 2^14, and a product is hi hi + lo hi
// + hi lo in fp32.  Against 64 bits the result is closer than the fp32 MFMA's,
// whose chains of 64 and more roundings are longer (8 steps of 32 terms here).
//
// Scales need the magnitudes within 2^12 of each other: V rows of one kv head
// (their scale is shared across the whole sum), and K and V rows of a tile;
// the columns of a tile within 2^16 (a column of small values is a dim of the
// output, or meets large ones of q: 2^20 apart it had 4.4e-6 in place of 1.3e-6);
// and everything finite and below 2^40, V rows not below 2^-41.  attn_split_prep records what it saw
// of a tile; a query block that meets anything else runs the fp32 form.
//
//  1. attn_split_prep: RoPE / norm of the new K rows as attn_prefill_prep, and
//     all rows 0 .. start + T of K and V as fp16 planes in MFMA operand order.
//  2. attn_split_flash: a workgroup takes a chunk of a query block's key
//     tiles, longest first, so the causal triangle and a short prompt over a
//     long cache load every CU alike.  A block of one chunk is finished there;
//     parts of others go to the workspace.
//  3. attn_split_merge: combines the parts.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int ST = 32;                       // key rows a tile
constexpr int SFRAGS = 64;                   // 1 KiB operand fragments a tile: 32 K, 32 V
constexpr int SPREP = 512, SWAVES = 8;
constexpr int LDO = kHd + 4;                 // padded LDS row stride of the output rows
// Largest workspace the split form takes (a sequence's planes are as large as
// its K and V rows); calls past it take the fp32 form.
constexpr size_t kSplitMaxBytes = (size_t)2 << 30;
constexpr int kScaleTop = 14, kPTop = 10, kMinExp = -40, kMaxExp = 40, kMaxSpread = 12, kMaxColSpread = 16;

// What attn_split_prep saw in a tile of one kv head.
struct TileMeta {
    float kdesc;          // 2^(ek - 14): K = (hi + lo) kdesc
    int ev;               // exponent of V's largest value: V = (hi + lo) 2^(ev - 14)
    int ev_min;           // exponent of the smallest nonzero row of V (kMaxExp: none)
    int bad;              // a value outside the range above
};

__device__ __forceinline__ uint32_t abs_bits(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// Exponent e with |x| < 2^e, x >= 2^(e-1), of a value's absolute bits.
__device__ __forceinline__ int exp_of(uint32_t bits) { return max((int)(bits >> 23) - 126, kMinExp); }

__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = max(h[0], h[1]);
    const auto q = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max(q[0], q[1]);
    v = max(v, row_xor_bits<8>(v));
    v = max(v, row_xor_bits<4>(v));
    v = max(v, row_xor_bits<2>(v));
    return max(v, row_xor_bits<1>(v));
}

__device__ __forceinline__ float pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// Workgroup: one 32-row tile of one kv head.  Wave a + 4 half holds its rows 16
// half + 4a .. + 3, half of the eight keys that lane group a of a V operand
// takes: 11.6 us for 2048 rows and 24.2 for 8133 (all eight rows in four
// waves: 13.7 and 27.5).
__global__ __launch_bounds__(SPREP) void attn_split_prep(
    const float* __restrict__ knew, const float* __restrict__ vnew, const float* __restrict__ k_norm, float* __restrict__ K,
    float* __restrict__ V, const float* __restrict__ rope_cos, const float* __restrict__ rope_sin,
    uint4* __restrict__ planes, TileMeta* __restrict__ meta, int start, int T, int nkv, int cap, float eps) {
    __shared__ uint4 frag[SFRAGS][64];
    __shared__ uint32_t red[8][4], colexp[8][2][64];
    __shared__ int badcol[2];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int a = wave & 3, half = wave >> 2;
    const int len = start + T, ntile = (len + ST - 1) / ST;
    const int tile = blockIdx.x / nkv, kvh = blockIdx.x % nkv, kv_dim = nkv * kHd;
    float4 kx[4], vx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = ST * tile + 16 * half + 4 * a + i;
        const size_t row = ((size_t)kvh * cap + p) * kHd + 4 * lane;
        const size_t nrow = (size_t)(p - start) * kv_dim + kvh * kHd + 4 * lane;
        kx[i] = vx[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p < len) {
            kx[i] = *reinterpret_cast<const float4*>(p < start ? K + row : knew + nrow);
            vx[i] = *reinterpret_cast<const float4*>(p < start ? V + row : vnew + nrow);
        }
    }
    // Largest absolute value of the tile's K and V, smallest nonzero row's.
    uint32_t kmax = 0, vmax = 0, kmin = ~0u, vmin = ~0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = ST * tile + 16 * half + 4 * a + i;
        if (p >= start && p < len) {
            const size_t row = ((size_t)kvh * cap + p) * kHd + 4 * lane;
            kx[i] = rope_norm_row(kx[i], lane, rope_cos + (size_t)p * kRopeHalf, rope_sin + (size_t)p * kRopeHalf, k_norm,
                                  eps, 1.0f);
            *reinterpret_cast<float4*>(K + row) = kx[i];
            *reinterpret_cast<float4*>(V + row) = vx[i];
        }
        const uint32_t mk = wave_umax(max(max(abs_bits(kx[i].x), abs_bits(kx[i].y)), max(abs_bits(kx[i].z), abs_bits(kx[i].w))));
        const uint32_t mv = wave_umax(max(max(abs_bits(vx[i].x), abs_bits(vx[i].y)), max(abs_bits(vx[i].z), abs_bits(vx[i].w))));
        kmax = max(kmax, mk);
        vmax = max(vmax, mv);
        if (mk) kmin = min(kmin, mk);
        if (mv) vmin = min(vmin, mv);
    }
    if (lane == 0) {
        red[wave][0] = kmax; red[wave][1] = vmax; red[wave][2] = kmin; red[wave][3] = vmin;
    }
    // The biased exponents of the largest values of the lane's four columns.
    auto exps = [](const float4 (&x)[4]) {
        auto top = [](float a, float b, float c, float d) {
            return max(max(abs_bits(a), abs_bits(b)), max(abs_bits(c), abs_bits(d))) >> 23;
        };
        return top(x[0].x, x[1].x, x[2].x, x[3].x) | top(x[0].y, x[1].y, x[2].y, x[3].y) << 8 |
               top(x[0].z, x[1].z, x[2].z, x[3].z) << 16 | top(x[0].w, x[1].w, x[2].w, x[3].w) << 24;
    };
    colexp[wave][0][lane] = exps(kx);
    colexp[wave][1][lane] = exps(vx);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        kmax = max(kmax, red[w][0]);
        vmax = max(vmax, red[w][1]);
        kmin = min(kmin, red[w][2]);
        vmin = min(vmin, red[w][3]);
    }
    const int ek = exp_of(kmax), ev = exp_of(vmax), ekm = kmin == ~0u ? ek : exp_of(kmin);
    const int evm = vmin == ~0u ? kMaxExp : exp_of(vmin);      // (rows of zeros have no place in the spread)
    // (V below the range of exp_of would be lost; small K only bring scores near 0.)
    const bool tiny = vmin != ~0u && (int)(vmin >> 23) - 126 < kMinExp;
    const bool bad = ek > kMaxExp || ev > kMaxExp || ek - ekm > kMaxSpread || tiny;
    // Waves 0 and 1: K's and V's smallest nonzero column.  (A tile of one row
    // has only its own values.)
    if (wave < 2) {
        int low = 255;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            int e = 0;
#pragma unroll
            for (int w = 0; w < 8; ++w) e = max(e, (int)((colexp[w][wave][lane] >> (8 * c)) & 255));
            if (e) low = min(low, e);
        }
        low = 255 - (int)wave_umax((uint32_t)(255 - low));
        if (lane == 0) badcol[wave] = len - ST * tile > 1 && (int)((wave ? vmax : kmax) >> 23) - low > kMaxColSpread;
    }
    const float ks = pow2(kScaleTop - min(ek, kMaxExp)), vs = pow2(kScaleTop - min(ev, kMaxExp));

    // Fragments as the flash kernel's operands: 16 bytes a lane (c16, g).  K,
    // fragment (16-row half, 32-dim step, plane): row c16, dims 8 g .. + 7 of
    // the step.  V, fragment 32 + (16-dim block, plane): dim c16, the keys of
    // wave g.  Slot c of a fragment sits at c ^ swz(fragment) in LDS (bank
    // spread of the stores below); the copy out undoes it.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c16 = 4 * a + i;
        const int step = lane >> 3, g = (lane >> 1) & 3;
        const float x[4] = {kx[i].x * ks, kx[i].y * ks, kx[i].z * ks, kx[i].w * ks};
        f16x4 hi, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            hi[j] = (_Float16)x[j];
            lo[j] = (_Float16)(x[j] - (float)hi[j]);
        }
        const int f = (half * 8 + step) * 2, c = (16 * g + c16) ^ step;
        reinterpret_cast<f16x4*>(&frag[f][c])[lane & 1] = hi;
        reinterpret_cast<f16x4*>(&frag[f + 1][c])[lane & 1] = lo;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f16x4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = (j == 0 ? vx[i].x : j == 1 ? vx[i].y : j == 2 ? vx[i].z : vx[i].w) * vs;
            hi[i] = (_Float16)x;
            lo[i] = (_Float16)(x - (float)hi[i]);
        }
        const int db = lane >> 2, f = 32 + 2 * db, c = (16 * a + 4 * (lane & 3) + j) ^ db;
        reinterpret_cast<f16x4*>(&frag[f][c])[half] = hi;
        reinterpret_cast<f16x4*>(&frag[f + 1][c])[half] = lo;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        meta[(size_t)kvh * ntile + tile] = TileMeta{pow2(min(ek, kMaxExp) - kScaleTop), ev, evm, bad || badcol[0] || badcol[1]};
    uint4* dst = planes + ((size_t)kvh * ntile + tile) * SFRAGS * 64;
#pragma unroll 4
    for (int f = wave; f < SFRAGS; f += 8) dst[64 * f + lane] = frag[f][lane ^ (f < 32 ? (f >> 1) & 7 : (f >> 1) & 15)];
}

// Shape of one split launch.  A query block's key tiles go in chunks of
// `chunk` from tile 0; an item is one chunk of one block, for every head group.
struct SplitPlan {
    int start, T, nh, nkv, hg;
    int rows;             // query rows a block: 16 (8 / hg), 16 of one head a wave
    int nqb, ntile, groups;
    int chunk, maxch;     // tiles a chunk, chunks of the longest block
    int items;            // items a head group
    int first_multi;      // first query block of more than one chunk
    bool listed;          // items in SplitItems, longest first; else block by block, longest first
    __host__ __device__ int tiles(int qb) const {
        const int r = rows * (qb + 1);
        return (start + (r < T ? r : T) + ST - 1) / ST;
    }
};
constexpr int kMaxItems = 512;
struct SplitItems { uint16_t v[kMaxItems]; };    // query block | chunk << 10

__device__ __forceinline__ f32x4 mfma_h(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// A part's floats in the workspace: O as each wave's registers, then (m, l) a lane.
constexpr size_t kPartFloats = (size_t)SWAVES * 64 * 64 + (size_t)SWAVES * 64 * 2;

__device__ __forceinline__ float4 gated(float4 o, float4 gate) {
    return make_float4(o.x * sigmoid_full(gate.x), o.y * sigmoid_full(gate.y), o.z * sigmoid_full(gate.z),
                       o.w * sigmoid_full(gate.w));
}

// Slot of a block's chunk in the parts.
__device__ __forceinline__ size_t part_slot(const SplitPlan& P, int qb, int c, int y) {
    return (((size_t)(qb - P.first_multi) * P.maxch + c) * P.groups + y) * kPartFloats;
}

// One item a workgroup: wave = q head hg y + wave % hg, 16 query rows wave /
// hg of the block, with its q rows (RoPE and norm as rope_norm_row, then split)
// and output accumulators in registers and the tiles, two buffers of 64 KiB,
// shared by the eight waves.  A step (one tile) is 96 MFMAs and 64 KiB of LDS
// reads a wave and takes 2.9 us; the matrix pipes are busy 36 % of the kernel's
// SIMD cycles at T = 2048, 47 % of those in which a CU has work, the rest is the
// softmax and the operand reads in front of each product.  T = 2048 behind
// nothing 122-129 us (fp32 MFMA 315), T = 4096 370 (1175), T = 133 behind 8000
// rows 70 (1085, 36 workgroups).  32 rows a wave, one wave a SIMD, halves the
// LDS reads but moves registers to and from the accumulation file: 508 us at
// T = 4096.
__global__ __launch_bounds__(64 * SWAVES, 2) void attn_split_flash(
    const uint4* __restrict__ planes, const TileMeta* __restrict__ meta, QRows Q, const float* __restrict__ K,
    const float* __restrict__ V, int cap, float* __restrict__ out, float* __restrict__ parts, int* __restrict__ fp32_done,
    SplitPlan P, SplitItems items) {
    // K and V operands of two tiles (128 KiB), or the fp32 form's tiles, or the
    // waves' output rows.
    __shared__ union {
        struct { uint4 k[2][SFRAGS / 2][64], v[2][SFRAGS / 2][64]; } t;
        Tiles fp32[2];
        float rows[SWAVES][16][LDO];
    } lds;
    __shared__ int red[4][SWAVES];
    const float* q_gate = Q.q_gate;
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroups of a head group share XCDs (block b runs on XCD b % 8), whose
    // L2 then holds the tiles that the group's workgroups read side by side.
    int y, r;
    if (8 % P.groups == 0) {
        const int per = 8 / P.groups, b = blockIdx.x;
        y = (b & 7) / per;
        r = (b >> 3) * per + (b & 7) % per;
    } else {
        y = blockIdx.x % P.groups;
        r = blockIdx.x / P.groups;
    }
    if (r >= P.items) return;
    int qb, c;
    if (P.listed) {
        qb = items.v[r] & 1023;
        c = items.v[r] >> 10;
    } else {
        qb = P.nqb - 1 - r / P.maxch;
        c = r % P.maxch;
    }
    const int n = P.tiles(qb), t0 = c * P.chunk, t1 = min(n, t0 + P.chunk);
    if (t0 >= t1) return;
    const int kvh = y * P.hg / (P.nh / P.nkv);
    planes += (size_t)kvh * P.ntile * SFRAGS * 64;
    meta += (size_t)kvh * P.ntile;

    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint4*>(planes), 0, (int)((uint32_t)P.ntile * (SFRAGS * 1024)), 0x00020000);
    auto stage = [&](uint4 (*dst)[64], int t, int first) {
#pragma unroll
        for (int i = 0; i < SFRAGS / 2 / SWAVES; ++i) {
            const int f = SWAVES * i + wave;
            dma_b128(prs, &dst[f][0], 16u * lane, (uint32_t)t * (SFRAGS * 1024) + 1024u * (first + f));
        }
    };
    auto stage_k = [&](int t) { stage(lds.t.k[(t - t0) & 1], t, 0); };
    auto stage_v = [&](int t) { stage(lds.t.v[(t - t0) & 1], t, SFRAGS / 2); };
    const int h = P.hg * y + wave % P.hg, row = P.rows * qb + 16 * (wave / P.hg) + c16;

    // q rows: lane (c16, g) holds dims 32 k + 8 g .. + 7, k < 8, of row c16.
    f16x8 qh[8], ql[8];
    float qdesc;
    const int qrow = min(P.T - 1, row), my_len = P.start + qrow + 1;
    bool bad;
    stage_k(t0);
    if (t0 + 1 < t1) stage_k(t0 + 1);
    stage_v(t0);
    {
        const int pos = P.start + qrow;
        const float* src = q_gate + ((size_t)qrow * P.nh + h) * 2 * kHd + 8 * g;
        const float* cs = Q.rope_cos + (size_t)pos * kRopeHalf + 8 * g;
        const float* sn = Q.rope_sin + (size_t)pos * kRopeHalf + 8 * g;
        float x[8][8];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float4 v = *reinterpret_cast<const float4*>(src + 32 * (i >> 1) + 4 * (i & 1));
            x[i >> 1][4 * (i & 1)] = v.x; x[i >> 1][4 * (i & 1) + 1] = v.y;
            x[i >> 1][4 * (i & 1) + 2] = v.z; x[i >> 1][4 * (i & 1) + 3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float co = cs[j], si = sn[j], x0 = x[0][j], x1 = x[1][j];
            x[0][j] = x0 * co - x1 * si;
            x[1][j] = x0 * si + x1 * co;
        }
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            float sk = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) sk += x[k][j] * x[k][j];
            ss += sk;
        }
        ss = xor16_sum(ss);
        ss = xor32_sum(ss);
        const float scale = 1.0f / sqrtf(ss / 256.0f + Q.eps), post = 1.0f / sqrtf((float)kHd);
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x[k][j] = x[k][j] * scale * (1.0f + Q.q_norm[32 * k + 8 * g + j]) * post;
                m = max(m, abs_bits(x[k][j]));
            }
        const auto mh = __builtin_amdgcn_permlane32_swap(m, m, false, false);
        m = max(mh[0], mh[1]);
        const auto mq = __builtin_amdgcn_permlane16_swap(m, m, false, false);
        m = max(mq[0], mq[1]);
        const int eq = min(exp_of(m), kMaxExp);
        bad = exp_of(m) > kMaxExp;
        const float qs = pow2(kScaleTop - eq);
        qdesc = pow2(eq - kScaleTop);
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float v = x[k][j] * qs;
                const _Float16 hi = (_Float16)v;
                qh[k][j] = hi;
                ql[k][j] = (_Float16)(v - (float)hi);
            }
    }
    // The V scale of the sum, the largest exponent of the tiles that the block
    // reads; and whether they are within the split's range, the same for all
    // of a block's chunks.
    int evmax = kMinExp;
    {
        int evmin = kMaxExp;
        for (int i = tid; i < n; i += 64 * SWAVES) {
            evmax = max(evmax, meta[i].ev);
            evmin = min(evmin, meta[i].ev_min);
            bad |= meta[i].bad != 0;
        }
        evmax = (int)wave_umax((uint32_t)(evmax + 1024)) - 1024;
        evmin = 1024 - (int)wave_umax((uint32_t)(1024 - evmin));
        const bool any = __any(bad);
        if (lane == 0) {
            red[0][wave] = evmax;
            red[1][wave] = evmin;
            red[2][wave] = any;
        }
        __syncthreads();
        int b = 0;
#pragma unroll
        for (int w = 0; w < SWAVES; ++w) {
            evmax = max(evmax, red[0][w]);
            evmin = min(evmin, red[1][w]);
            b |= red[2][w];
        }
        bad = b || evmax - evmin > kMaxSpread;
    }
    if (c == 0 && tid == 0 && n > P.chunk) fp32_done[(qb - P.first_multi) * P.groups + y] = bad;
    if (bad) {
        // The block's rows in two halves, one to each of its first two chunks'
        // workgroups (133 tokens behind 8000 rows of 4 q heads a kv head 1150
        // us, of one 1162; all in the first chunk's, 16 rows after another, 2299
        // and 9078; the fp32 kernels alone 1090), or one to each half of a
        // single chunk's (64 tokens 47, one after the other 62; 25).
        const int subs = 4 / P.hg, nch = (n + P.chunk - 1) / P.chunk;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (nch == 1)
            flash_fp32_block<false>(lds.fp32, Q, K, V, out, P.start, P.T, P.nh, P.nkv, P.hg, cap, qb, y, subs);
        else if (c < 2 && (2 * qb + c) * subs * QR < P.T)
            flash_fp32_block<true>(lds.fp32, Q, K, V, out, P.start, P.T, P.nh, P.nkv, P.hg, cap, 2 * qb + c, y, subs);
        return;
    }

    // S^T of keys 32 t + 16 half + 4 g + r, query c16, less its scale: hi hi,
    // and the two cross products.
    struct Scores { f32x4 hh[2], x[2]; };
    auto scores = [&](int t) {
        Scores S = {};
        const f16x8* F = reinterpret_cast<const f16x8*>(&lds.t.k[(t - t0) & 1][0][lane]);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            f16x8 kh[2], kl[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                kh[i] = F[64 * ((8 * i + k) * 2)];
                kl[i] = F[64 * ((8 * i + k) * 2 + 1)];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) S.hh[i] = mfma_h(kh[i], qh[k], S.hh[i]);
#pragma unroll
            for (int i = 0; i < 2; ++i) S.x[i] = mfma_h(kl[i], qh[k], S.x[i]);
#pragma unroll
            for (int i = 0; i < 2; ++i) S.x[i] = mfma_h(kh[i], ql[k], S.x[i]);
        }
        return S;
    };
    // A column's running maximum is below every score the split's range
    // allows until its first unmasked position (P = 0 up to there).
    float m_run = -1e30f, l_run = 0.0f;
    f32x4 O[16];
#pragma unroll
    for (int db = 0; db < 16; ++db) O[db] = {0.f, 0.f, 0.f, 0.f};
    // A step holds tile t's softmax and P V and tile t + 1's scores.  The two
    // waves of a SIMD (w, w + 4) take them in opposite orders, so one's VALU
    // work and LDS waits run beside the other's MFMAs.
    Scores S = {};
    // t1 hidden from the optimizer: where it sees that a step always stages the
    // next tile, it waits for those loads before it reads the tile it has.
    int te = t1;
    asm volatile("" : "+s"(te));
    auto step = [&](int t, auto first, auto more, auto masked) {
        const TileMeta mt = meta[t];
        // K of tile t + 1 and V of tile t have landed and every wave is past
        // tile t - 1; the next ones go out.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        if (t + 2 < te) stage_k(t + 2);
        if (t + 1 < te) stage_v(t + 1);
        const float sc = qdesc * mt.kdesc;
        float st[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float v = (S.hh[i][q] + S.x[i][q]) * sc;
                st[i][q] = !masked || ST * t + 16 * i + 4 * g + q < my_len ? v : -INFINITY;
            }
        if constexpr (first && more) {
            S = scores(t + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // The reference point moves only when a score passes it by e^3.4 < 2^5
        // (P then stays below 2^15).
        float mx = m_run;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) mx = fmaxf(mx, st[i][q]);
        if (__any(mx - m_run > 3.4f)) {
            mx = xor16_max(mx);
            mx = xor32_max(mx);
            const float alpha = __expf(m_run - mx);
            m_run = mx;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < 16; ++db) O[db] = O[db] * alpha;
        }
        // P in units of 2^(evmax - ev - kPTop), O in units of 2^(evmax - kPTop - 14).
        const float ps = pow2(max(kPTop + min(mt.ev, kMaxExp) - evmax, -100));
        f16x8 ph, pl;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float e = __expf(st[i][q] - m_run);
                l_run += e;                    // this lane's keys; the column's sum at the end
                const float p = e * ps;
                const _Float16 hi = (_Float16)p;
                ph[4 * i + q] = hi;
                pl[4 * i + q] = (_Float16)(p - (float)hi);
            }
        // O^T += V^T P^T
        const f16x8* F = reinterpret_cast<const f16x8*>(&lds.t.v[(t - t0) & 1][0][lane]);
#pragma unroll
        for (int d4 = 0; d4 < 4; ++d4) {
            f16x8 vh[4], vl[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                vh[d] = F[64 * (2 * (4 * d4 + d))];
                vl[d] = F[64 * (2 * (4 * d4 + d) + 1)];
            }
#pragma unroll
            for (int d = 0; d < 4; ++d) O[4 * d4 + d] = mfma_h(vl[d], ph, O[4 * d4 + d]);
#pragma unroll
            for (int d = 0; d < 4; ++d) O[4 * d4 + d] = mfma_h(vh[d], pl, O[4 * d4 + d]);
#pragma unroll
            for (int d = 0; d < 4; ++d) O[4 * d4 + d] = mfma_h(vh[d], ph, O[4 * d4 + d]);
        }
        if constexpr (!first && more) {
            __builtin_amdgcn_sched_barrier(0);
            S = scores(t + 1);
        }
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    S = scores(t0);
    // Tiles up to `open` lie before every row's own position.
    const int open = min(t1 - 1, (P.start + P.rows * qb + 1) / ST);
    auto run = [&](auto first) {
        int t = t0;
        for (; t < open; ++t) step(t, first, std::true_type{}, std::false_type{});
        for (; t + 1 < t1; ++t) step(t, first, std::true_type{}, std::true_type{});
        step(t, first, std::false_type{}, std::true_type{});
    };
    if (wave < 4) run(std::true_type{});
    else run(std::false_type{});
    l_run = xor16_sum(l_run);
    l_run = xor32_sum(l_run);
    if (n <= P.chunk) {
        // The item's rows go through LDS (the tiles', once every wave is past
        // them) and on to the waves in turn, so that a gate load and a store
        // cover a whole row and a few rows share all waves; four rows a step,
        // in a loop, as code that runs once costs its fetch (stored from the
        // accumulators' own lanes, a call of one token took 6 us more).
        const float inv = pow2(evmax - kPTop - kScaleTop) / l_run;
        const int hs = __builtin_ctz(P.hg), t_base = P.rows * qb, n_rows = min(P.rows, P.T - t_base) << hs;
        struct RowAt { size_t at; int lds; };
        auto row_at = [&](int step, int i) {
            const int q = min(wave + SWAVES * (4 * step + i), n_rows - 1), t = q >> hs, hh = q & (P.hg - 1);
            return RowAt{((size_t)(t_base + t) * P.nh + P.hg * y + hh) * kHd, (((t >> 4) * P.hg + hh) * 16 + (t & 15)) * LDO};
        };
        float4 gate[4];
        auto load_gates = [&](int step) {
#pragma unroll
            for (int i = 0; i < 4; ++i) gate[i] = *reinterpret_cast<const float4*>(q_gate + 2 * row_at(step, i).at + kHd + 4 * lane);
        };
        load_gates(0);
        lds_barrier();
#pragma unroll
        for (int db = 0; db < 16; ++db)
            *reinterpret_cast<f32x4*>(&lds.rows[wave][c16][16 * db + 4 * g]) = O[db] * inv;
        lds_barrier();
        const float* rows = &lds.rows[0][0][0];
#pragma unroll 1
        for (int step = 0; wave + SWAVES * 4 * step < n_rows; ++step) {
            const float4 now[4] = {gate[0], gate[1], gate[2], gate[3]};
            load_gates(step + 1);
            float4 o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = *reinterpret_cast<const float4*>(rows + row_at(step, i).lds + 4 * lane);
            // The first position (a wave's first row) attends to itself alone: its V as it is.
            if (P.start + t_base + step == 0 && wave < P.hg)
                o[0] = *reinterpret_cast<const float4*>(V + (size_t)kvh * cap * kHd + 4 * lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o[i] = gated(o[i], now[i]);
                if (wave + SWAVES * (4 * step + i) < n_rows) *reinterpret_cast<float4*>(out + row_at(step, i).at + 4 * lane) = o[i];
            }
        }
    } else {
        float* po = parts + part_slot(P, qb, c, y);
#pragma unroll
        for (int db = 0; db < 16; ++db)
            reinterpret_cast<float4*>(po)[(wave * 16 + db) * 64 + lane] = make_float4(O[db][0], O[db][1], O[db][2], O[db][3]);
        reinterpret_cast<float2*>(po + (size_t)SWAVES * 64 * 64)[wave * 64 + lane] = make_float2(m_run, l_run);
    }
}

// Four 16-dim blocks of one flash wave's rows of a query block, combined over
// the block's chunks: wave w takes chunks w, w + 4, .., then wave 0 the four.
__global__ __launch_bounds__(256) void attn_split_merge(const TileMeta* __restrict__ meta, const float* __restrict__ parts,
                                                        const int* __restrict__ fp32_done, const float* __restrict__ q_gate,
                                                        float* __restrict__ out, SplitPlan P) {
    __shared__ float4 xo[3][4][64];
    __shared__ float2 xml[3][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
    const int d4 = blockIdx.x & 3, wave = blockIdx.x >> 2, y = blockIdx.y, qb = P.first_multi + blockIdx.z;
    const int row0 = P.rows * qb + 16 * (wave / P.hg), row = row0 + c16;
    const int h = P.hg * y + wave % P.hg;
    if (row0 >= P.T || fp32_done[blockIdx.z * P.groups + y]) return;
    const int kvh = y * P.hg / (P.nh / P.nkv), n = P.tiles(qb), nch = (n + P.chunk - 1) / P.chunk;
    float m = -1e30f, l = 0.0f;
    f32x4 o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](float2 ml, const float4 (&x)[4]) {
        const float mx = fmaxf(m, ml.x);
        const float f0 = __expf(m - mx), f1 = __expf(ml.x - mx);
        m = mx;
        l = l * f0 + ml.y * f1;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            o[d][0] = o[d][0] * f0 + x[d].x * f1;
            o[d][1] = o[d][1] * f0 + x[d].y * f1;
            o[d][2] = o[d][2] * f0 + x[d].z * f1;
            o[d][3] = o[d][3] * f0 + x[d].w * f1;
        }
    };
#pragma unroll 2
    for (int c = w; c < nch; c += 4) {
        const float* p = parts + part_slot(P, qb, c, y);
        const float2 ml = reinterpret_cast<const float2*>(p + (size_t)SWAVES * 64 * 64)[wave * 64 + lane];
        float4 x[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) x[d] = reinterpret_cast<const float4*>(p)[(wave * 16 + 4 * d4 + d) * 64 + lane];
        add(ml, x);
    }
    if (w > 0) {
#pragma unroll
        for (int d = 0; d < 4; ++d) xo[w - 1][d][lane] = make_float4(o[d][0], o[d][1], o[d][2], o[d][3]);
        xml[w - 1][lane] = make_float2(m, l);
    }
    int ev = kMinExp;
    if (w == 0) {
        for (int i = lane; i < n; i += kWave) ev = max(ev, meta[(size_t)kvh * P.ntile + i].ev);
        ev = min((int)wave_umax((uint32_t)(ev + 1024)) - 1024, kMaxExp);
    }
    __syncthreads();
    if (w > 0 || row >= P.T) return;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        float4 x[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) x[d] = xo[i][d][lane];
        add(xml[i][lane], x);
    }
    const float inv = pow2(ev - kPTop - kScaleTop) / l;
    const float* grow = q_gate + ((size_t)row * P.nh + h) * 2 * kHd + kHd + 64 * d4 + 4 * g;
    float* orow = out + ((size_t)row * P.nh + h) * kHd + 64 * d4 + 4 * g;
    float4 gate[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) gate[d] = *reinterpret_cast<const float4*>(grow + 16 * d);
#pragma unroll
    for (int d = 0; d < 4; ++d)
        *reinterpret_cast<float4*>(orow + 16 * d) =
            gated(make_float4(o[d][0] * inv, o[d][1] * inv, o[d][2] * inv, o[d][3] * inv), gate[d]);
}

}  // namespace

namespace {

// Parts of a head group's chunked query blocks at most (no plan that the shares
// ask for has more: 30000 shapes).
long max_parts(const SplitPlan& p, int slots) { return p.nqb < slots ? 2L * slots : slots; }

// Chunks from the share of one workgroup a CU, longer until the items of more
// than half a chunk fit the CUs once (two of them would share one).
SplitPlan plan_split(const Dims& d, int n_cu, int start, int T) {
    SplitPlan p{};
    p.start = start;
    p.T = T;
    p.nh = d.nh;
    p.nkv = d.nkv;
    const int g = d.nh / d.nkv;
    p.hg = g < 4 ? g : 4;
    p.rows = 16 * (SWAVES / p.hg);
    p.nqb = (T + p.rows - 1) / p.rows;
    p.ntile = (start + T + ST - 1) / ST;
    p.groups = d.nh / p.hg;
    const int slots = std::max(1, n_cu / p.groups);
    long total = 0;
    for (int q = 0; q < p.nqb; ++q) total += p.tiles(q);
    int chunk = (int)std::max<long>((total + slots - 1) / slots, 4);
    if (p.nqb >= 2 * slots) chunk = p.ntile;
    chunk = std::max(chunk, (p.ntile + 63) / 64);              // the item list's 6 bits
    for (; chunk < p.ntile; chunk += std::max(1, chunk / 32)) {
        int big = 0, multi = 0;
        for (int q = 0; q < p.nqb; ++q) {
            const int n = p.tiles(q);
            big += n / chunk + (2 * (n % chunk) > chunk);
            multi += n > chunk;
        }
        if (big <= slots && (long)multi * ((p.ntile + chunk - 1) / chunk) <= max_parts(p, slots)) break;
    }
    p.chunk = std::min(chunk, p.ntile);
    p.maxch = (p.ntile + p.chunk - 1) / p.chunk;
    p.first_multi = p.nqb;
    while (p.first_multi > 0 && p.tiles(p.first_multi - 1) > p.chunk) --p.first_multi;
    p.items = 0;
    for (int q = 0; q < p.nqb; ++q) p.items += (p.tiles(q) + p.chunk - 1) / p.chunk;
    p.listed = p.items <= kMaxItems && p.nqb <= 1024;
    if (!p.listed) p.items = p.nqb * p.maxch;
    return p;
}

// The items by length, longest first; equal ones chunk by chunk.
void list_items(const SplitPlan& p, SplitItems& it) {
    int k = 0;
    std::array<uint32_t, kMaxItems> key;
    for (int q = 0; q < p.nqb; ++q)
        for (int c = 0; c * p.chunk < p.tiles(q); ++c) {
            const int len = std::min(p.tiles(q) - c * p.chunk, p.chunk);
            key[k++] = ((uint32_t)(0xffff - std::min(len, 0xffff)) << 16) | (uint32_t)(c << 10) | (uint32_t)q;
        }
    std::sort(key.begin(), key.begin() + k);
    for (int i = 0; i < k; ++i) it.v[i] = (uint16_t)key[i];
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Workspace of the split form.
struct SplitWork {
    size_t fp32_done, meta, planes, parts, bytes;
    explicit SplitWork(const SplitPlan& p) {
        fp32_done = 0;
        meta = align256((size_t)(p.nqb - p.first_multi) * p.groups * sizeof(int));
        planes = align256(meta + (size_t)p.nkv * p.ntile * sizeof(TileMeta));
        parts = align256(planes + (size_t)p.nkv * p.ntile * SFRAGS * 1024);
        bytes = parts + (size_t)(p.nqb - p.first_multi) * p.maxch * p.groups * kPartFloats * sizeof(float);
    }
};

// Workspace of any split call of T tokens on this context: one of its
// capacity, so that it is allocated once and not again as a sequence grows
// (nor under a stream capture after one call of as many tokens).
size_t split_reserve(const q35m_ctx* c, const SplitPlan& p) {
    const int slots = std::max(1, c->n_cu / p.groups);
    const long ntile = ((long)c->cap + ST - 1) / ST, chunks = (ntile + 3) / 4;
    const long parts = chunks > 1 && p.nqb < 2 * slots ? std::min<long>(max_parts(p, slots), p.nqb * chunks) : 0;
    const size_t bytes = align256((size_t)p.nqb * p.groups * sizeof(int)) + align256((size_t)p.nkv * ntile * sizeof(TileMeta)) +
                         (size_t)p.nkv * ntile * SFRAGS * 1024 + (size_t)parts * p.groups * kPartFloats * sizeof(float) + 768;
    return std::min(bytes, kSplitMaxBytes);
}

// Whether the call takes the split form, with its workspace in place.  A size
// that could not be had is not asked for again.
bool split_ready(q35m_ctx* c, const SplitPlan& p, size_t bytes) {
    // A kv head's planes are addressed through one buffer descriptor.
    if ((size_t)p.ntile * SFRAGS * 1024 > c->tile_limit || bytes > kSplitMaxBytes) return false;
    for (const size_t n : {std::max(bytes, split_reserve(c, p)), bytes}) {
        if (n <= c->work_bytes) return true;
        if (n >= c->split_refused) continue;
        if (ensure_work(c, n) == hipSuccess) return true;
        (void)hipGetLastError();
        c->split_refused = n;
    }
    return false;
}

}  // namespace

hipError_t launch_attn_prefill(q35m_ctx* c, int layer, int seq, int start, int T,
                               const float* q_gate, const float* k, const float* v, float* out) {
    const Dims& d = c->d;
    const AttnLayer& L = c->full[layer];
    float* K = L.k_cache + (size_t)seq * c->cap * d.kv_dim;
    float* V = L.v_cache + (size_t)seq * c->cap * d.kv_dim;
    const QRows Q{q_gate, L.q_norm, c->rope_cos, c->rope_sin, d.eps};
    // Head groups of up to 4 q heads of one kv head.
    const int g = d.nh / d.nkv, hg = g < 4 ? g : 4;
    const SplitPlan p = plan_split(d, c->n_cu, start, T);
    const SplitWork wk(p);
    if (split_ready(c, p, wk.bytes)) {
        char* base = reinterpret_cast<char*>(c->work);
        int* fp32_done = reinterpret_cast<int*>(base + wk.fp32_done);
        TileMeta* meta = reinterpret_cast<TileMeta*>(base + wk.meta);
        uint4* planes = reinterpret_cast<uint4*>(base + wk.planes);
        float* parts = reinterpret_cast<float*>(base + wk.parts);
        {
            ProfScope ps_(c, K_ATTN_SPLIT_PREP);
            hipExtLaunchKernelGGL(attn_split_prep, dim3(p.ntile * d.nkv), dim3(SPREP), 0, c->stream, ps_.a, ps_.b, 0, k, v,
                                  L.k_norm, K, V, c->rope_cos, c->rope_sin, planes, meta, start, T, d.nkv, c->cap, d.eps);
        }
        {
            SplitItems items;
            if (p.listed) list_items(p, items);
            const int per = 8 % p.groups == 0 ? 8 / p.groups : 1;
            ProfScope ps_(c, K_ATTN_SPLIT_FLASH);
            hipExtLaunchKernelGGL(attn_split_flash, dim3(p.groups * ((p.items + per - 1) / per * per)), dim3(64 * SWAVES), 0,
                                  c->stream, ps_.a, ps_.b, 0, planes, meta, Q, K, V, c->cap, out, parts, fp32_done, p, items);
        }
        if (p.first_multi < p.nqb) {
            ProfScope ps_(c, K_ATTN_SPLIT_MERGE);
            hipExtLaunchKernelGGL(attn_split_merge, dim3(4 * SWAVES, p.groups, p.nqb - p.first_multi), dim3(256), 0,
                                  c->stream, ps_.a, ps_.b, 0, meta, parts, fp32_done, q_gate, out, p);
        }
        return hipGetLastError();
    }
    {
        ProfScope ps_(c, K_ATTN_PREFILL_PREP);
        hipExtLaunchKernelGGL(attn_prefill_prep, dim3(T, d.nkv), dim3(kWave), 0, c->stream, ps_.a, ps_.b, 0, k, v, L.k_norm,
                              K, V, c->rope_cos, c->rope_sin, start, d.nkv, c->cap, d.eps);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    {
        ProfScope ps_(c, K_ATTN_PREFILL_FLASH);
        hipExtLaunchKernelGGL(attn_prefill_flash, dim3((T + QR - 1) / QR * (d.nh / hg)), dim3(512), 0,
                           c->stream, ps_.a, ps_.b, 0, Q, K, V, out, start, T, d.nh, d.nkv, hg, c->cap);
    }
    return hipGetLastError();
}

}  // namespace q35
