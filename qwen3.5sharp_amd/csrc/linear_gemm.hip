// Quantized projections of several tokens on the matrix cores.  The reference's
// result is exact integer sums per block or sub-block followed by fp32 chains
// in block order (linear_q.hip states the formats, the reference's functions,
// the one-token kernels and the tiles of many tokens of Q4_K and Q6_K):
//
//   Q4_K    per 32-value sub-block  acc = fma(sc_s dot_s, dw dx, acc); per block
//           mn = fma(sum_j min_j bsums, dmin dx, mn); acc - mn
//   Q6_K    per block and lane k < 8  acc_k = fma(dw dx, sumi_k, acc_k)
//   Q5_K    per block  acc += d (sum_s sc_s dot_s) - dmin (sum_j min_j bsums)
//   IQ4_XS  per 32-value sub-block  acc += (d (ls - 32) dot_s) dx
//   Q2_0C   per 256 values T; panel rows acc = fma(T, dw dx, acc), raw rows
//           per 512 values acc += dw (T0 dx0 + T1 dx1)
//   STQ1_0  per 256 values T; panel rows acc = fma(T, dw dx, acc), raw rows
//           acc += (dw dx) T
//
// (dots, sums and T exact integers, no fused multiply-add but where written), so
// results are the reference's bits at any tile shape.
//
// (linear_gemm_split, below, is the form for few outputs.)  A wave holds 16
// weight rows x 16 TT tokens.  The dots are int8 MFMAs: A is
// the tokens' Q8_K bytes from LDS, B the rows' values, decoded in registers
// from each lane's own share of its row (no LDS, no exchange between waves;
// the four lane groups of a row cover its block without overlap) and loaded
// two or more blocks ahead.  So per block a wave spends its decode once for
// all its token tiles, and per output one multiply-add a sub-block (Q5_K), or
// the chain's own operations.  The workgroup's waves share the tokens, CH
// blocks at a time through two LDS buffers filled by buffer loads straight
// into LDS while the other one is worked on.  Bound by instruction issue: Q5_K
// at 500 tokens of 2560 -> 8192 takes 451 VALU and 40 MFMA instructions a block
// of 16 rows x 64 tokens and issues on 68 % of all SIMD cycles, 84 % of those
// in which its CU has work.
#include <algorithm>

#include "common.h"
#include "q35mix_internal.h"
#include "quant_layout.h"

namespace q35 {
namespace {

// Rows of the 2-byte aligned formats are read at their own addresses.
typedef uint32_t u32_a2 __attribute__((aligned(2)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// A lane's share (lane group lg) of one 256-value block of its row.
template <int QT> struct RowBlock;

template <> struct RowBlock<4> {       // header; qs bytes 8 lg .. + 7 of each 32
    uint4 hdr;
    uint2 qs[4];
    __device__ __forceinline__ void load(const unsigned char* row, int b, int lg) {
        const unsigned char* p = row + (size_t)b * Q4K_BYTES;
        hdr = *reinterpret_cast<const uint4*>(p);
#pragma unroll
        for (int j = 0; j < 4; ++j) qs[j] = *reinterpret_cast<const uint2*>(p + 16 + 32 * j + 8 * lg);
    }
};

// Half lg / 2 of ql and qh, the scales and d, as the dwords from the 4-byte
// boundary below the 2-byte aligned block (16-byte loads at 2-byte aligned
// addresses cost 1.5-2.7 us more a call); the rows of a launch end on a 4-byte
// boundary.
template <> struct RowBlock<6> {
    uint32_t ql[17], qh[9], sc[5];
    uint32_t sh;
    __device__ __forceinline__ void load(const unsigned char* row, int b, int lg) {
        const size_t at = reinterpret_cast<size_t>(row) + (size_t)b * Q6K_BYTES;
        const unsigned char* p = reinterpret_cast<const unsigned char*>(at & ~(size_t)3);
        const int j = lg >> 1;
        sh = (uint32_t)at & 3;
        words<17>(ql, p + 64 * j);
        words<9>(qh, p + 128 + 32 * j);
        words<5>(sc, p + 192);
    }
    template <int N> static __device__ __forceinline__ void words(uint32_t (&v)[N], const unsigned char* p) {
#pragma unroll
        for (int i = 0; i + 4 <= N; i += 4) {
            const u32x4_a4 x = *reinterpret_cast<const u32x4_a4*>(p + 4 * i);
            v[i] = x[0]; v[i + 1] = x[1]; v[i + 2] = x[2]; v[i + 3] = x[3];
        }
        v[N - 1] = *reinterpret_cast<const uint32_t*>(p + 4 * (N - 1));
    }
};

template <> struct RowBlock<5> {       // header; qh and qs bytes 8 lg .. + 7 of each 32
    uint4 hdr;
    uint2 qh, qs[4];
    __device__ __forceinline__ void load(const unsigned char* row, int b, int lg) {
        const unsigned char* p = row + (size_t)b * Q5K_BYTES;
        hdr = *reinterpret_cast<const uint4*>(p);
        qh = *reinterpret_cast<const uint2*>(p + 16 + 8 * lg);
#pragma unroll
        for (int j = 0; j < 4; ++j) qs[j] = *reinterpret_cast<const uint2*>(p + 48 + 32 * j + 8 * lg);
    }
};

template <> struct RowBlock<14> {      // header; bytes 8 (lg % 2) .. + 7 of each sub-block's 16
    uint2 hdr, qs[8];
    __device__ __forceinline__ void load(const unsigned char* row, int b, int lg) {
        const unsigned char* p = row + (size_t)b * IQ4XS_BYTES;
        hdr = *reinterpret_cast<const uint2*>(p);
#pragma unroll
        for (int s = 0; s < 8; ++s) qs[s] = *reinterpret_cast<const uint2*>(p + 8 + 16 * s + 8 * (lg & 1));
    }
};

template <> struct RowBlock<2> {       // d; the 4 code bytes of values 64 s + 16 lg .. + 15
    uint32_t d, qs[4];
    __device__ __forceinline__ void load(const unsigned char* row, int b, int lg) {
        const unsigned char* p = row + (size_t)(b >> 1) * Q2_BYTES;
        d = *reinterpret_cast<const uint16_t*>(p);
#pragma unroll
        for (int s = 0; s < 4; ++s) qs[s] = *reinterpret_cast<const u32_a2*>(p + 2 + 64 * (b & 1) + 16 * s + 4 * lg);
    }
};

template <> struct RowBlock<1> {       // d; slots and signs of chunk lg (16 groups)
    uint32_t d, sign;
    u32x2_a2 qs;
    __device__ __forceinline__ void load(const unsigned char* row, int b, int lg) {
        const unsigned char* p = row + (size_t)b * STQ_BYTES;
        qs = *reinterpret_cast<const u32x2_a2*>(p + 8 * lg);
        sign = *reinterpret_cast<const uint16_t*>(p + 32 + 2 * lg);
        d = *reinterpret_cast<const uint16_t*>(p + 40);
    }
};

// v of the four 16-lane groups, in every lane.
__device__ __forceinline__ void lane_groups(uint32_t v, uint32_t (&r)[4]) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
    r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
}

// Terms of the fp32 chain a block adds to an output: (a, b) pairs, in order.
template <int QT> constexpr int kTerms = QT == 4 ? 9 : QT == 14 || QT == 6 ? 8 : 1;

// The running values of 16 rows x 16 TT tokens: lane (l16, lg) holds tokens
// 16 tt + 4 lg + r of weight row l16 (the layout of an MFMA result).  v[1]:
// Q4_K's min sum, or a raw Q2_0C row's first product of a 512-value pair;
// v[0..7]: Q6_K's lanes.
template <int QT> constexpr int kAccs = QT == 6 ? 8 : QT == 4 || QT == 2 ? 2 : 1;
template <int QT, int TT> struct Acc {
    float v[kAccs<QT>][TT][4];
    __device__ __forceinline__ float result(int tt, int r) const {
#pragma clang fp contract(off)
        if constexpr (QT == 4) {
            return v[0][tt][r] - v[1][tt][r];
        } else if constexpr (QT == 6) {    // VecDotQ4K.HorizontalSum (VecDotQ4K.cs:145-151)
            const float s0 = v[0][tt][r] + v[4][tt][r], s1 = v[1][tt][r] + v[5][tt][r];
            const float s2 = v[2][tt][r] + v[6][tt][r], s3 = v[3][tt][r] + v[7][tt][r];
            return (s0 + s2) + (s1 + s3);
        } else {
            return v[0][tt][r];
        }
    }
};

// Term s of a block in the reference's chain.
template <int QT, int TT>
__device__ __forceinline__ void chain(Acc<QT, TT>& acc, int s, int tt, int r, float a, float b, int blk, bool panel) {
#pragma clang fp contract(off)
    float& v = acc.v[QT == 6 ? s : QT == 4 ? s >> 3 : 0][tt][r];
    if constexpr (QT == 4 || QT == 6) {
        v = fmaf(a, b, v);
    } else if constexpr (QT == 5 || QT == 14) {
        v = v + a;
    } else if (panel) {
        v = fmaf(a, b, v);
    } else if constexpr (QT == 1) {
        v = v + b * a;
    } else {
        float& pend = acc.v[QT == 2 ? 1 : 0][tt][r];
        if (blk & 1) v = v + b * (pend + a);
        else pend = a;
    }
}

// One block of 16 rows x 16 TT tokens: forms its chain terms and hands each to
// term(s, tt, r, a, b), for every output in ascending s.  X: the block's
// tokens in LDS, Q8K_WORDS apart.
template <int QT, int TT, typename F>
__device__ __forceinline__ void block_terms(const RowBlock<QT>& w, const uint32_t* X, int l16, int lg, bool panel, F&& term) {
#pragma clang fp contract(off)
    const uint32_t* xa = X + l16 * Q8K_WORDS;                    // A rows: token 16 tt + l16
    auto dx = [&](int tt, int r) { return __builtin_bit_cast(float, X[(16 * tt + 4 * lg + r) * Q8K_WORDS]); };
    const i32x4 zero = {0, 0, 0, 0};
    // Q4_K / Q5_K min sum of a token tile, sum_j min_j (bsums 2j, 2j + 1): j =
    // lg and lg + 4 of this lane's row (B) and token (A); at most 8 x 63 x
    // 4064, exact in fp32.
    auto min_sum = [&](int tt, uint32_t S1, uint32_t S2) {
        const float m0 = (float)((S1 >> (8 * lg)) & 63);
        const float m1 = (float)(((S2 >> (8 * lg + 4)) & 15) | (((S1 >> (8 * lg + 6)) & 3) << 4));
        const uint32_t* xb = xa + 16 * tt * Q8K_WORDS + Q8K_BS;
        float pa[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t p = xb[lg + 4 * h];
            pa[h] = (float)((int)(int16_t)(p & 0xffff) + (int)(int16_t)(p >> 16));
        }
        const f32x4 md = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[0], m0, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x4f32(pa[1], m1, md, 0, 0, 0);
    };
    if constexpr (QT == 4) {
        // The dot starts at the bits of 1.5 * 2^23 and is read as fp32, so that
        // fma(dot, sc, -1.5 * 2^23 sc) = sc dot exactly (as in q4k_gemm).
        const int m = 0x4B400000;
        const i32x4 magic = {m, m, m, m};
        const uint32_t S0 = w.hdr.y, S1 = w.hdr.z, S2 = w.hdr.w;
        const uint32_t sl = S0 & 0x3f3f3f3fu, sh = (S2 & 0x0f0f0f0fu) | ((S0 >> 2) & 0x30303030u);
        const float dw = half_bits_to_float(w.hdr.x & 0xffff), dmw = half_bits_to_float(w.hdr.x >> 16);
        float cs[TT][4];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) cs[tt][r] = dw * dx(tt, r);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t q0 = w.qs[s >> 1].x, q1 = w.qs[s >> 1].y;
            const uint32_t b0 = ((s & 1) ? q0 >> 4 : q0) & 0x0f0f0f0fu, b1 = ((s & 1) ? q1 >> 4 : q1) & 0x0f0f0f0fu;
            const long bv = (long)(((unsigned long)b1 << 32) | b0);
            const float scf = (float)(((s < 4 ? sl : sh) >> (8 * (s & 3))) & 0xffu), negc = scf * -12582912.0f;
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const long av = *reinterpret_cast<const long*>(xa + 16 * tt * Q8K_WORDS + Q8K_QS + 8 * s + 2 * lg);
                const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, magic, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) term(s, tt, r, fmaf(__int_as_float(d[r]), scf, negc), cs[tt][r]);
            }
        }
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            const f32x4 md = min_sum(tt, S1, S2);
#pragma unroll
            for (int r = 0; r < 4; ++r) term(8, tt, r, md[r], dmw * dx(tt, r));
        }
    } else if constexpr (QT == 6) {
        // Lane k's sum as two planes of one 16x16x64 product each (the notes
        // at q6k_gemm in linear_q.hip): lane group lg brings parts (j, m0),
        // (j, m0 + 1) at bytes 4k .. + 3 and the bsums term.
        const int j = lg >> 1, odd = lg & 1;
        auto at = [&](const uint32_t* v, int i) { return __builtin_amdgcn_alignbyte(v[i + 1], v[i], w.sh); };
        const float dw = half_bits_to_float((w.sc[4] >> (8 * w.sh)) & 0xffff);
        float d[TT][4];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) d[tt][r] = dx(tt, r) * dw;
        const uint32_t rq = odd ? 3 : 31, rh0 = odd ? 31 : 27, rh1 = odd ? 1 : 29;
        const uint32_t sc4[4] = {at(w.sc, 0), at(w.sc, 1), at(w.sc, 2), at(w.sc, 3)};
        const uint32_t scw = lg < 2 ? (lg ? sc4[1] : sc4[0]) : (lg & 1 ? sc4[3] : sc4[2]);   // scales 4 lg .. + 3
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t qa = at(w.ql, k), qb = at(w.ql, 8 + k), qh = at(w.qh, k);
            const uint32_t v0 = (__builtin_amdgcn_alignbit(qa, qa, rq) & 0x1e1e1e1eu) |
                                (__builtin_amdgcn_alignbit(qh, qh, rh0) & 0x60606060u);
            const uint32_t v1 = (__builtin_amdgcn_alignbit(qb, qb, rq) & 0x1e1e1e1eu) |
                                (__builtin_amdgcn_alignbit(qh, qh, rh1) & 0x60606060u);
            uint32_t l0, h0, l1, h1;
            q6k_split(v0, (int)(int8_t)(scw >> (8 * (k >> 2))), l0, h0);
            q6k_split(v1, (int)(int8_t)(scw >> (8 * (2 + (k >> 2)))), l1, h1);
            // -32 scales[2k + j] = 128 ((-s) >> 2) + 32 ((-s) & 3), bytes replicated
            const int neg = -(int)(int8_t)(sc4[k >> 1] >> (16 * (k & 1) + 8 * j));
            const uint32_t elo = __builtin_amdgcn_perm(0u, (uint32_t)((neg & 3) << 5), 0u);
            const uint32_t ehi = __builtin_amdgcn_perm(0u, (uint32_t)(neg >> 2), 0u);
            const i32x4 bh = {(int)h0, (int)h1, (int)ehi, (int)ehi}, bl = {(int)l0, (int)l1, (int)elo, (int)elo};
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const uint32_t* xt = xa + 16 * tt * Q8K_WORDS + Q8K_QS;
                const int qv = 32 * j + 16 * odd + k, qe = 8 * k + 4 * j + 2 * odd;
                const i32x4 av = {(int)xt[qv], (int)xt[qv + 8], (int)xt[qe], (int)xt[qe + 1]};
                const i32x4 dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bh, zero, 0, 0, 0);
                const i32x4 dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bl, zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) term(k, tt, r, d[tt][r], (float)((int)((unsigned)dh[r] << 7) + dl[r]));
            }
        }
    } else if constexpr (QT == 5) {
        const uint32_t S0 = w.hdr.y, S1 = w.hdr.z, S2 = w.hdr.w;
        const uint32_t sl = S0 & 0x3f3f3f3fu;                                  // scales 0-3
        const uint32_t sh = (S2 & 0x0f0f0f0fu) | ((S0 >> 2) & 0x30303030u);    // scales 4-7
        int isum[TT][4];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) isum[tt][r] = 0;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            auto val = [&](uint32_t q, uint32_t h) {
                const uint32_t h4 = s < 4 ? h << (4 - s) : h >> (s - 4);       // qh bit s to bit 4
                return (((s & 1) ? q >> 4 : q) & 0x0f0f0f0fu) | (h4 & 0x10101010u);
            };
            const uint32_t b0 = val(w.qs[s >> 1].x, w.qh.x), b1 = val(w.qs[s >> 1].y, w.qh.y);
            const long bv = (long)(((unsigned long)b1 << 32) | b0);
            const int sc = (int)(((s < 4 ? sl : sh) >> (8 * (s & 3))) & 0xffu);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const long av = *reinterpret_cast<const long*>(xa + 16 * tt * Q8K_WORDS + Q8K_QS + 8 * s + 2 * lg);
                const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    isum[tt][r] += __mul24(d[r], sc);
                    // one multiply-add each (summed in pairs it takes three operations for two)
                    asm volatile("" : "+v"(isum[tt][r]));
                }
            }
        }
        const float dw = half_bits_to_float(w.hdr.x & 0xffff), dmw = half_bits_to_float(w.hdr.x >> 16);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            const f32x4 md = min_sum(tt, S1, S2);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float yd = dx(tt, r), d = dw * yd, dmin = dmw * yd;
                term(0, tt, r, d * (float)isum[tt][r] - dmin * md[r], 0.0f);
            }
        }
    } else if constexpr (QT == 14) {
        const float d = half_bits_to_float(w.hdr.x & 0xffff);
        const uint32_t sh = 4 * (lg >> 1);                       // low or high nibbles
        float yd[TT][4];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) yd[tt][r] = dx(tt, r);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t b0 = iq4_grid((w.qs[s].x >> sh) & 0x0f0f0f0fu), b1 = iq4_grid((w.qs[s].y >> sh) & 0x0f0f0f0fu);
            const long bv = (long)(((unsigned long)b1 << 32) | b0);
            const int ls = (int)(((w.hdr.y >> (8 * (s >> 1) + 4 * (s & 1))) & 0xf) | (((w.hdr.x >> (16 + 2 * s)) & 3) << 4));
            const float dl = d * (float)(ls - 32);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const long av = *reinterpret_cast<const long*>(xa + 16 * tt * Q8K_WORDS + Q8K_QS + 8 * s + 2 * lg);
                const i32x4 dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) term(s, tt, r, dl * (float)dot[r] * yd[tt][r], 0.0f);
            }
        }
    } else {
        i32x4 t[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) t[tt] = zero;
        uint32_t pat[4][4];            // STQ1_0: [i][chunk]
        if constexpr (QT == 1)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                lane_groups(stq_patterns((w.qs[i >> 1] >> (16 * (i & 1))) & 0xffffu, (w.sign >> (4 * i)) & 0xfu), pat[i]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            i32x4 bv;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (QT == 1) {
                    // lane lg of each pattern, less 1
                    bv[i] = (int)__builtin_amdgcn_perm(0u, 0x020100FFu, (pat[i][s] >> (2 * lg)) & 0x03030303u);
                } else {
                    // the byte's four codes spread over four bytes, then 2 code - 3
                    const uint32_t c = (w.qs[s] >> (8 * i)) & 0xffu, c2 = c | (c << 12);
                    bv[i] = (int)__builtin_amdgcn_perm(0u, 0x0301FFFDu, (c2 | (c2 << 6)) & 0x03030303u);
                }
            }
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const i32x4 av = *reinterpret_cast<const i32x4*>(xa + 16 * tt * Q8K_WORDS + Q8K_QS + 16 * s + 4 * lg);
                t[tt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, t[tt], 0, 0, 0);
            }
        }
        const float dw = half_bits_to_float(w.d);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float T = (float)t[tt][r], x = dx(tt, r);
                if (QT == 1 || panel) term(0, tt, r, T, dw * x);
                else term(0, tt, r, T * x, dw);
            }
    }
}

template <int QT>
__host__ __device__ constexpr size_t row_bytes(int nb) {
    return QT == 4 ? (size_t)nb * Q4K_BYTES : QT == 6 ? (size_t)nb * Q6K_BYTES : QT == 5 ? (size_t)nb * Q5K_BYTES : QT == 14 ? (size_t)nb * IQ4XS_BYTES : QT == 2 ? (size_t)(nb >> 1) * Q2_BYTES
                                                                                            : (size_t)nb * STQ_BYTES;
}

template <int QT, int TT>
__device__ __forceinline__ void store_tile(const Acc<QT, TT>& acc, float* y, int row, int n_rows, int n_out, int tok0,
                                           int tokens, int lg) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = tok0 + 16 * tt + 4 * lg + r;
            if (row < n_rows && t < tokens) y[(size_t)t * n_out + row] = acc.result(tt, r);
        }
}

// Blocks of the tokens in one LDS buffer: two buffers are 76 KiB, two
// workgroups a CU.
template <int TT> constexpr int kChunk = 8 / TT;

template <int QT, int TT, int NW>
__global__ __launch_bounds__(64 * NW) void linear_gemm(const unsigned char* __restrict__ w, const uint32_t* __restrict__ q8,
                                                       float* __restrict__ y, int n_in, int n_rows, int n_out, int tokens,
                                                       int panel_rows) {
    constexpr int TOK = 16 * TT, CH = kChunk<TT>, PF = CH < 4 ? CH : 4;
    constexpr int XW = Q8K_WORDS / 4;                            // 16-byte pieces of a Q8_K block
    constexpr int RUNS = (TOK * XW + 63) / 64;                   // wave-wide loads of one block's tokens
    __shared__ uint4 xsh[2][CH][TOK * XW];
    const int nb = n_in / QK;
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = (blockIdx.x * NW + wave) * 16, tok0 = blockIdx.y * TOK;
    const int row = row0 + l16;
    const unsigned char* wrow = w + (size_t)min(row, n_rows - 1) * row_bytes<QT>(nb);
    const bool panel = row < panel_rows;

    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(q8), 0, (int)((uint32_t)tokens * nb * Q8K_WORDS * 4), 0x00020000);
    auto stage = [&](int b0, int buf) {
        for (int u = wave; u < CH * RUNS; u += NW) {
            const int k = u / RUNS, q = u % RUNS, i = 64 * q + lane, b = b0 + k;
            const uint32_t vo = (uint32_t)min(tok0 + i / XW, tokens - 1) * nb * Q8K_WORDS * 4 + 16 * (i % XW);
            if (b < nb && i < TOK * XW) dma_b128(xrs, &xsh[buf][k][64 * q], vo, (uint32_t)b * Q8K_WORDS * 4);
        }
    };
    RowBlock<QT> wq[PF];
#pragma unroll
    for (int u = 0; u < PF; ++u) wq[u].load(wrow, min(u, nb - 1), lg);
    Acc<QT, TT> acc = {};

    stage(0, 0);
    for (int b0 = 0, buf = 0; b0 < nb; b0 += CH, buf ^= 1) {
        // This chunk's tokens have landed, and every wave is past the last one.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (b0 + CH < nb) stage(b0 + CH, buf ^ 1);
#pragma unroll 1
        for (int k0 = 0; k0 < CH; k0 += PF)
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int k = k0 + u, b = b0 + k;
                if (b < nb) {
                    // The next load goes out before the block's work: the chunk's
                    // closing wait covers it.
                    const RowBlock<QT> wb = wq[u];
                    wq[u].load(wrow, min(b + PF, nb - 1), lg);
                    block_terms<QT, TT>(wb, reinterpret_cast<const uint32_t*>(xsh[buf][k]), l16, lg, panel,
                                        [&](int s, int tt, int r, float a, float f) { chain<QT, TT>(acc, s, tt, r, a, f, b, panel); });
                }
            }
    }
    store_tile(acc, y, row, n_rows, n_out, tok0, tokens, lg);
}

// The same for few outputs (few tokens, or few rows): a workgroup takes 16 RG
// rows x 16 TT tokens and its waves split the blocks, KW at a time, wave (rg,
// kw) forming block p KW + kw's terms.  The chain then passes from wave to
// wave in block order through LDS, a barrier a step.
constexpr int kSplitWaves = 10;

template <int QT, int TT, int RG>
__global__ __launch_bounds__(64 * kSplitWaves) void linear_gemm_split(const unsigned char* __restrict__ w,
                                                                      const uint32_t* __restrict__ q8, float* __restrict__ y,
                                                                      int n_in, int n_rows, int n_out, int tokens,
                                                                      int panel_rows, int KW) {
    constexpr int TOK = 16 * TT, XW = Q8K_WORDS / 4, XB = TOK * XW, RUNS = (XB + 63) / 64;
    constexpr int NT = kTerms<QT>, NV = kAccs<QT>;
    extern __shared__ uint4 split_smem[];                        // two buffers of KW blocks' tokens, then the chain
    const int nb = n_in / QK, passes = (nb + KW - 1) / KW;
    const int lane = threadIdx.x & 63, l16 = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kw = wave % KW, rg = wave / KW;
    const int row = (blockIdx.x * RG + rg) * 16 + l16, tok0 = blockIdx.y * TOK;
    const unsigned char* wrow = w + (size_t)min(row, n_rows - 1) * row_bytes<QT>(nb);
    const bool panel = row < panel_rows;
    float4* relay = reinterpret_cast<float4*>(split_smem + (passes > 1 ? 2 : 1) * KW * XB) + rg * NV * TT * 64 + lane;

    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(q8), 0, (int)((uint32_t)tokens * nb * Q8K_WORDS * 4), 0x00020000);
    // A row group's share of block b's tokens (past the last token: not loaded, not stored).
    const int nchunk = min(tokens - tok0, TOK) * XW;
    auto stage = [&](int b, int buf) {
        if (b >= nb) return;
#pragma unroll
        for (int q0 = 0; q0 < RUNS; q0 += RG) {
            const int q = q0 + rg, i = 64 * q + lane;
            if (i < nchunk)
                dma_b128(xrs, split_smem + (buf * KW + kw) * XB + 64 * q,
                         (uint32_t)(tok0 + i / XW) * nb * Q8K_WORDS * 4 + 16 * (i % XW), (uint32_t)b * Q8K_WORDS * 4);
        }
    };
    RowBlock<QT> wn;
    wn.load(wrow, min(kw, nb - 1), lg);
    stage(kw, 0);
    Acc<QT, TT> acc = {};
    for (int p = 0; p < passes; ++p) {
        const int b = p * KW + kw;
        // This pass's tokens have landed, and every wave is past the last one's.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const RowBlock<QT> wb = wn;
        if (p + 1 < passes) {
            stage(b + KW, (p + 1) & 1);
            wn.load(wrow, min(b + KW, nb - 1), lg);
        }
        float ta[NT][TT][4], tb[NT][TT][4];
        if (b < nb)
            block_terms<QT, TT>(wb, reinterpret_cast<const uint32_t*>(split_smem + ((p & 1) * KW + kw) * XB), l16, lg, panel,
                                [&](int s, int tt, int r, float a, float f) { ta[s][tt][r] = a; tb[s][tt][r] = f; });
        const int steps = min(KW, nb - p * KW);
        if constexpr (QT == 6) {
            // Eight chains an output: every wave's terms to LDS, and each wave
            // then runs its share of the lanes over the pass's blocks (passed
            // from wave to wave, the chains took 0.4 us a block).
            static_assert(TT == 1 && RG == 1, "one tile a workgroup");
            if (b < nb) {
#pragma unroll
                for (int s = 0; s < 8; ++s) relay[(kw * 9 + s) * 64] = *reinterpret_cast<const float4*>(tb[s][0]);
                relay[(kw * 9 + 8) * 64] = *reinterpret_cast<const float4*>(ta[0][0]);
            }
            lds_barrier();
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (s % KW == kw)
#pragma unroll 4
                    for (int k = 0; k < steps; ++k) {
                        const float4 x = relay[(k * 9 + s) * 64], d = relay[(k * 9 + 8) * 64];
                        chain<QT, TT>(acc, s, 0, 0, d.x, x.x, b, panel);
                        chain<QT, TT>(acc, s, 0, 1, d.y, x.y, b, panel);
                        chain<QT, TT>(acc, s, 0, 2, d.z, x.z, b, panel);
                        chain<QT, TT>(acc, s, 0, 3, d.w, x.w, b, panel);
                    }
            if (p + 1 < passes) continue;
            lds_barrier();
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (s % KW == kw) relay[s * 64] = *reinterpret_cast<const float4*>(acc.v[s][0]);
            lds_barrier();
            if (kw > 0) return;
#pragma unroll
            for (int s = 0; s < 8; ++s) *reinterpret_cast<float4*>(acc.v[s][0]) = relay[s * 64];
            store_tile(acc, y, row, n_rows, n_out, tok0, tokens, lg);
            continue;
        }
        for (int k = 0; k < steps; ++k) {
            if (kw == k) {
                if (b > 0)
#pragma unroll
                    for (int i = 0; i < NV * TT; ++i) *reinterpret_cast<float4*>(acc.v[i / TT][i % TT]) = relay[64 * i];
#pragma unroll
                for (int s = 0; s < NT; ++s)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) chain<QT, TT>(acc, s, tt, r, ta[s][tt][r], tb[s][tt][r], b, panel);
                if (b + 1 < nb) {
#pragma unroll
                    for (int i = 0; i < NV * TT; ++i) relay[64 * i] = *reinterpret_cast<const float4*>(acc.v[i / TT][i % TT]);
                } else {
                    store_tile(acc, y, row, n_rows, n_out, tok0, tokens, lg);
                }
            }
            if (k + 1 < steps) lds_barrier();
        }
    }
}

template <int QT>
hipError_t go(q35m_ctx* c, int kid, const unsigned char* w, const uint32_t* q8, float* y, int n_in, int n_rows, int n_out,
              int tokens, int panel_rows) {
    const int nb = n_in / QK;
    auto pieces = [&](int tok, auto one) {
        // The tokens are addressed through a buffer descriptor: at most 2 GiB a launch.
        const size_t lim = (c->tile_limit - 1) / ((size_t)nb * Q8K_WORDS * 4) / tok * tok;
        const int tmax = (int)std::min<size_t>(tokens, std::max<size_t>(lim, tok));
        for (int t0 = 0; t0 < tokens; t0 += tmax) {
            const int nt = std::min(tmax, tokens - t0);
            ProfScope ps_(c, kid);
            one(ps_, q8 + (size_t)t0 * nb * Q8K_WORDS, y + (size_t)t0 * n_out, nt);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    };
    auto whole = [&](auto kern, int tok, int nw) {
        return pieces(tok, [&](ProfScope& ps, const uint32_t* qt, float* yt, int nt) {
            hipExtLaunchKernelGGL(kern, dim3((n_rows + 16 * nw - 1) / (16 * nw), (nt + tok - 1) / tok), dim3(64 * nw), 0,
                                  c->stream, ps.a, ps.b, 0, w, qt, yt, n_in, n_rows, n_out, nt, panel_rows);
        });
    };
    auto split = [&](auto kern, int tt, int rg) {
        // Q6_K: two passes' tokens and the terms of eight waves fill the LDS.
        const int wmax = QT == 6 && nb > kSplitWaves ? 8 : kSplitWaves / rg;
        const int passes = (nb + wmax - 1) / wmax, kw = (nb + passes - 1) / passes;
        const size_t chains = QT == 6 ? (size_t)std::max(kw * 9, 8) : (size_t)rg * kAccs<QT> * tt;
        const size_t lds = ((passes > 1 ? 2 : 1) * (size_t)kw * tt * 16 * Q8K_WORDS / 4 + chains * 64) * 16;
        return pieces(16 * tt, [&](ProfScope& ps, const uint32_t* qt, float* yt, int nt) {
            hipExtLaunchKernelGGL(kern, dim3((n_rows + 16 * rg - 1) / (16 * rg), (nt + 16 * tt - 1) / (16 * tt)),
                                  dim3(64 * kw * rg), lds, c->stream, ps.a, ps.b, 0, w, qt, yt, n_in, n_rows, n_out, nt,
                                  panel_rows, kw);
        });
    };
    // By the 16 x 16 tiles of the result.  Few: every tile its own workgroup,
    // the blocks split over its waves; then pairs of them; then waves that
    // run whole rows of blocks, of 32 and of 64 tokens (least decode a token,
    // but a serial 3 us a block where the waves are few).  Measured (us, in
    // that order; 2560 -> 8192 unless said): Q5_K 16 tokens (512 tiles) 7.9 /
    // 9.9 / 19 / 32, 32 (1024) 16 / 10.4 / 19 / 32, 64 (2048) 27 / 17.3 / 22 /
    // 33, 128 (4096) 48 / 33 / 22 / 33, 500 177 / 127 / 61 / 48, 2048 tokens -
    // / 500 / 218 / 170; 4096 -> 2560 at 64 tokens (640) 14.9 / 14.7 / 30 /
    // 51, at 200 (2080) 36 / 29 / 32 / 51; IQ4_XS at 200 (6656) - / 67 / 46 /
    // 35; Q2_0C at 200 - / 57 / 26 / 19.  One thread a block and a serial
    // chain a row for 8 tokens at a time took 7.1 at 2 tokens, 17.6 at 16, 310
    // at 500, 1246 at 2048 (IQ4_XS 373, Q2_0C 422, STQ1_0 770 at 500).
    const long tiles = (long)((n_rows + 15) / 16) * ((tokens + 15) / 16);
    if constexpr (QT == 6) {
        return split(linear_gemm_split<QT, 1, 1>, 1, 1);
    } else {
        // Q4_K at 16 tokens 10.9 / 9.3 / 18 / 25, at 64 34 / 17.6 / 18 / 25, at
        // 128 66 / 32 / 19 / 26, at 256 131 / 63 / 34 / 27; 2560 -> 1024 at 64
        // tokens (256 tiles) 6.8 / 9.7 / 18 / 24; 512 -> 12288 at 96 (4608) - / -
        // / 15 / 11.
        if (tiles <= (QT == 4 ? 400 : 640)) return split(linear_gemm_split<QT, 1, 1>, 1, 1);
        if (tiles <= (QT == 4 ? 1536 : 2304)) return split(linear_gemm_split<QT, 2, 2>, 2, 2);
        // (Up to 32 tokens fill no 64: 2560 -> 151936 at 8 tokens 78 / 113; rows
        // of two blocks hardly load: 512 -> 151936 28 / 20 for Q2_0C.)
        if (tiles <= (QT == 4 ? 4096 : 4608) || (tokens <= 32 && nb > 2)) return whole(linear_gemm<QT, 2, 8>, 32, 8);
        return whole(linear_gemm<QT, 4, 8>, 64, 8);
    }
}

}  // namespace

hipError_t launch_linear_gemm(q35m_ctx* c, int qtype, const void* w, const void* q8, float* y, int n_in, int n_rows,
                              int n_out, int tokens, int panel_rows) {
    const unsigned char* wb = reinterpret_cast<const unsigned char*>(w);
    const uint32_t* qb = reinterpret_cast<const uint32_t*>(q8);
    switch (qtype) {
        case 4: return go<4>(c, K_Q4K_SMALL, wb, qb, y, n_in, n_rows, n_out, tokens, 0);
        case 6: return go<6>(c, K_Q6K_SMALL, wb, qb, y, n_in, n_rows, n_out, tokens, 0);
        case 5: return go<5>(c, K_Q5K_GEMM, wb, qb, y, n_in, n_rows, n_out, tokens, 0);
        case 14: return go<14>(c, K_IQ4XS_GEMM, wb, qb, y, n_in, n_rows, n_out, tokens, 0);
        case 2: return go<2>(c, K_Q2_0C_GEMM, wb, qb, y, n_in, n_rows, n_out, tokens, panel_rows);
        default: return go<1>(c, K_STQ1_0_GEMM, wb, qb, y, n_in, n_rows, n_out, tokens, panel_rows);
    }
}

}  // namespace q35
