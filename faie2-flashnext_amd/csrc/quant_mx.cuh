// The GEMV on the bf16 matrix cores (k_gemv_mx, k_gemv_mx_grp): templates of the quant_mx*.hip units.
//
// y[t][r] = sum_j W[r][j] x[t][j] for up to 8 tokens is a product of a 16-row weight tile with a thin x.  On the VALU
// (quant_impl.cuh) every weight costs its decode and one multiply-add a token; here it costs its decode alone, and the
// products of all tokens go to v_mfma_f32_16x16x32_bf16:
//
//   * weights: every format's codes are small integers (or the bf16 values themselves), exact in bf16.  The group's
//     scale multiplies the 32-value dot product afterwards, in fp32, as on the VALU.
//   * x: an fp32 value is the exact sum of three bf16 values (hi = its first 8 significant bits, mid the next 8, lo
//     the last 8), so that every product is exact and the sums are fp32: nothing of x is rounded away.  (Values too
//     small for bf16 to hold all three are scaled by a power of two first, MxX::split.)
//   * tile: x is the A operand, 16 rows = 4 tokens x {hi, mid, lo, unused}; 16 weight rows are the B operand.  Lane
//     (r, c) = (lane % 16, lane / 16) of the result holds hi, mid and lo of token c for weight row r, so that the
//     scale, the sum of the three and the accumulator are one lane's: no shuffle anywhere.
//   * operand layout: lane (r, c) loads 16-byte pieces of row r's quants (4 lanes read 64 consecutive bytes) and a
//     4 x 4 exchange across the lane quarters (4 v_permlane swaps for 4 words) hands each lane word c of every piece.
//
// Work split: a workgroup walks 16-row tiles; its waves split the row, UPW units of 256 values each (a unit of a
// K-quant is a super-block), and keep their slice of x in registers for all tiles (split once, through 3 KB of LDS
// of the wave's own).  The waves' partial sums of a tile meet in LDS, summed in wave order.  Which values a wave sums
// depends on the columns alone, never on the rows, the tokens, the grid or a group, so token t of an nt-token call
// gets the bits of a one-token call, and a weight of a grouped launch those of its own.
//
// What bounds it: at one token the launch, x's round trip and split and the weight's first round trip (about 4 us, the
// whole of a small weight), then the decode.  By the counters of IQ4_XS 10240 x 2560 at 1 / 8 tokens: 4.1 / 5.5 vector
// instructions a value, x's split included, the vector units busy 46 / 39 % of the time and the matrix cores 5 / 7 %.
// One weight decode serves all tokens of a call up to 4096 columns; wider rows (two units a wave) take 4 tokens at a
// time, so that a call of 5 to 8 reads and decodes the weight twice.
// Cold weights, us a call, the vector kernels / this, at 1, 4 and 8 tokens:
//   IQ4_XS 10240 x 2560     9.2 /  7.6   15.9 /  8.7   23.0 /  10.7
//   Q6_K    6144 x 2560     8.4 /  7.7   10.7 /  9.0   15.3 /  10.2
//   Q8_0    2560 x 6144     7.9 /  7.8   12.4 /  9.2   19.1 /  13.1
//   Q8_0    2048 x 4096     5.8 /  6.0    7.4 /  7.0    9.8 /   8.6
//   BF16      96 x 2560     4.4 /  4.0    5.8 /  4.8    8.3 /   5.9
//   IQ3_S    640 x 2560     5.6 /  5.1    6.9 /  5.9    9.6 /   7.1
//   Q4_K   20000 x 8192    25.4 / 21.6   46.0 / 23.6  122.6 /  37.6
//   Q5_K  248320 x 2560   109.9 /102.8  176.8 / 107.1  271.2 / 130.8
//   Q5_K    2560 x 8192     9.6 /  8.7   13.7 / 10.9   27.7 /  15.9
//   Q6_K   20000 x 8192    30.0 / 35.2   51.5 / 35.6  130.1 /  53.8
//   Q6_K     300 x 8192     6.5 /  7.3    9.8 /  9.4   19.3 /   9.6
//   grouped: DeltaNet's qkv, z (Q6_K), alpha and beta  13.3 / 11.8   23.4 / 12.9   33.3 / 15.6
//            attention's q, k, v and indexer           12.9 / 10.0   20.0 / 11.1   27.9 / 12.5
//            the FFN's router, shared gate and up       6.2 /  6.3    7.6 /  6.9    9.9 /  7.5
//            the same at 4096 columns                   6.8 /  7.6    8.4 /  8.3   10.7 /  9.4
// Error against 64 bits over 1024 to 6144 columns: 0.6 to 1.1e-7 (the vector kernels 0.8 to 1.1e-7), Q6_K 2.0e-7 (2.1e-7).
#pragma once

#include "quant_impl.cuh"

namespace fn {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));
struct __attribute__((packed)) U16p { uint32_t w[4]; };  // 16 bytes at any alignment

// a 4 x 4 exchange across the lane quarters: before, quarter q holds words 0..3 of piece q; after, it holds word q of
// pieces 0..3
__device__ __forceinline__ void quarter_exchange(uint32_t *w) {
    const auto s32 = [](uint32_t &a, uint32_t &b) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0], b = r[1];
    };
    const auto s16 = [](uint32_t &a, uint32_t &b) {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0], b = r[1];
    };
    s32(w[0], w[2]);
    s32(w[1], w[3]);
    s16(w[0], w[1]);
    s16(w[2], w[3]);
}

// the high halves (bf16) of two floats, a in the low half
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
__device__ __forceinline__ uint32_t pack_f(float a, float b) { return pack_hi(__float_as_uint(a), __float_as_uint(b)); }
// 8 codes 0 .. 255 as bf16 subnormals: the code in the low bits of a bf16 is code x 2^-133 (up to 255 the spacing does
// not change; the matrix cores take subnormal inputs exactly), so that unpacking a code is its byte and nothing else,
// no conversion.  Their x is scaled by a power of two (DEN below).  A format's codes sit at the top of the byte: the
// products are lined up by their exponents as they stand, so a code with leading zeros would lose that many of the
// sum's low bits (4-bit codes at the bottom of the byte: error 1.4e-6 instead of 1.4e-7 on an x with outliers).
__device__ __forceinline__ v4u codes(uint32_t a, uint32_t b) {
    return v4u{__builtin_amdgcn_perm(0u, a, 0x0C010C00u), __builtin_amdgcn_perm(0u, a, 0x0C030C02u),
               __builtin_amdgcn_perm(0u, b, 0x0C010C00u), __builtin_amdgcn_perm(0u, b, 0x0C030C02u)};
}
__device__ __forceinline__ float ubyte(uint32_t w, int k) { return (float) ((w >> (8 * k)) & 0xFFu); }
// 8 signed bytes as bf16
__device__ __forceinline__ v4u bytes_s(uint32_t a, uint32_t b) {
    v4u f;
    f.x = pack_f(sbyte(a, 0), sbyte(a, 1));
    f.y = pack_f(sbyte(a, 2), sbyte(a, 3));
    f.z = pack_f(sbyte(b, 0), sbyte(b, 1));
    f.w = pack_f(sbyte(b, 2), sbyte(b, 3));
    return f;
}

// Where the 8 values of lane quarter q sit in a group of 32 (the x fragments follow the weights' order):
//   HALVES: 4q .. 4q + 3, then 16 + 4q ..;  NIBBLES: 4q, 16 + 4q, 4q + 1, 17 + 4q, ...;  RUN: 8q .. 8q + 7
//   GRID: 8 p .. 8 p + 7, p = q with its two bits exchanged
enum { HALVES, NIBBLES, RUN, GRID };

// Per format: NW words of a unit (256 values of one row) in a lane, load() them (q = the lane's quarter), arrange()
// once per unit, then per group j of the unit frag() (8 values as bf16) and scale() (s, and m of the formats with a
// minimum).  SUB: two scales a group (16 values each, halves of a HALVES fragment).
//   MIN: the value is d (s q) - dm m with d, dm of the unit (super()); DEN: q are codes(), exact as subnormals, and x is
//   scaled so that a unit's largest |x| is just under 2^120: products of anything that counts are normal numbers.
template <uint32_t TY> struct MX;

template <> struct MX<QT_BF16> {
    static constexpr int NW = 32, MAP = RUN;
    static constexpr bool MIN = false, SUB = false, CHAIN = true, DEN = false;
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
#pragma unroll
        for (int j = 0; j < 4; ++j) ld16(R.b0 + (512 * u + 64 * j + 16 * q), w + 4 * j);
    }
    // (its other half apart: 32 words and the x being split do not fit 80 registers)
    template <class R_> __device__ static void load2(const R_ &R, int u, int q, uint32_t *w) {
#pragma unroll
        for (int j = 4; j < 8; ++j) ld16(R.b0 + (512 * u + 64 * j + 16 * q), w + 4 * j);
    }
    __device__ static void arrange(uint32_t *) {}
    __device__ static v4u frag(const uint32_t *w, int j, int, const uint8_t *) {
        return v4u{w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]};
    }
    __device__ static void scale(const uint32_t *, int, float *, float *) {}
};

template <> struct MX<QT_Q8_0> {
    static constexpr int NW = 20, MAP = HALVES;
    static constexpr bool MIN = false, SUB = false, CHAIN = false, DEN = false;
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) ld16(R.b0 + (256 * u + 64 * k + 16 * q), w + 4 * k);
        ld16(R.b1 + 16 * u, w + 16);
    }
    __device__ static void arrange(uint32_t *w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) quarter_exchange(w + 4 * k);
    }
    __device__ static v4u frag(const uint32_t *w, int j, int, const uint8_t *) { return bytes_s(w[2 * j], w[2 * j + 1]); }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *) {
        s[0] = h2f(w[16 + (j >> 1)] >> (16 * (j & 1)));
    }
};

// The 256 pairs of IQ4 levels that a byte's nibbles name, as bf16 pairs in LDS (low nibble in the low half), 32 copies
// of each: lane l reads copy l % 32, so that a wave's lookups never meet in a bank.  One lookup gives two values.
__device__ __forceinline__ void iq4_pairs_fill(uint8_t *tab, int tid, int nth) {
    const auto lev = [](uint32_t i) {
        const uint32_t kw = i < 8 ? (i < 4 ? KV0 : KV1) : (i < 12 ? KV2 : KV3);
        return (float) (int8_t) (kw >> (8 * (i & 3)));
    };
    // a thread writes one entry's 32 copies, or half of them when there are threads enough (nth >= 256); the pieces of
    // 16 bytes start at the entry's number, so that the lanes of a store cover the banks
    const uint32_t e = (uint32_t) tid & 255u;
    const int n = nth >= 512 ? 4 : 8, k0 = tid >> 8;
    if (tid >= (nth >= 512 ? 512 : 256)) return;
    const uint32_t v = pack_f(lev(e & 15u), lev(e >> 4));
    for (int k = 0; k < n; ++k) *reinterpret_cast<v4u *>(tab + 128 * e + 16 * ((e + n * k0 + k) & 7u)) = v4u{v, v, v, v};
}
__device__ __forceinline__ v4u iq4_pairs(uint32_t w, int lane, const uint8_t *tab) {
    const uint32_t at = 4u * ((uint32_t) lane & 31u);
    const auto ld = [&](uint32_t off) { return *reinterpret_cast<const uint32_t *>(tab + off); };
    return v4u{ld(((w << 7) & 0x7F80u) | at), ld(((w >> 1) & 0x7F80u) | at), ld(((w >> 9) & 0x7F80u) | at),
               ld(((w >> 17) & 0x7F80u) | at)};
}

template <> struct MX<QT_IQ4_NL> {
    static constexpr int NW = 12, MAP = NIBBLES;
    static constexpr bool MIN = false, SUB = false, CHAIN = false, DEN = false;
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
        ld16(R.b0 + (128 * u + 16 * q), w);
        ld16(R.b0 + (128 * u + 64 + 16 * q), w + 4);
        ld16(R.b1 + 16 * u, w + 8);
    }
    __device__ static void arrange(uint32_t *w) {
        quarter_exchange(w);
        quarter_exchange(w + 4);
    }
    __device__ static v4u frag(const uint32_t *w, int j, int lane, const uint8_t *tab) { return iq4_pairs(w[j], lane, tab); }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *) {
        s[0] = h2f(w[8 + (j >> 1)] >> (16 * (j & 1)));
    }
};

template <> struct MX<QT_IQ4_XS> {
    static constexpr int NW = 11, MAP = NIBBLES;
    static constexpr bool MIN = false, SUB = false, CHAIN = false, DEN = false;
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
        ld16(R.b0 + (128 * u + 16 * q), w);
        ld16(R.b0 + (128 * u + 64 + 16 * q), w + 4);
        ld8(R.b1 + 8 * u, w + 8);
    }
    __device__ static void arrange(uint32_t *w) {
        quarter_exchange(w);
        quarter_exchange(w + 4);
        // the 6-bit scales as bytes: of groups 0, 2, 4, 6 in w[9], of 1, 3, 5, 7 in w[10]
        const auto spread = [](uint32_t h) {  // 2 bits of every nibble of h to bits 4, 5 of a byte each
            h &= 0x3333u;
            h = (h | h << 8) & 0x00FF00FFu;
            return (h << 4 | h << 8) & 0x30303030u;
        };
        const uint32_t sl = w[9], sh = w[8] >> 16;
        w[9] = (sl & 0x0F0F0F0Fu) | spread(sh);
        w[10] = ((sl >> 4) & 0x0F0F0F0Fu) | spread(sh >> 2);
    }
    __device__ static v4u frag(const uint32_t *w, int j, int lane, const uint8_t *tab) { return iq4_pairs(w[j], lane, tab); }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *) {
        const float d = h2f(w[8]);  // (d (ls - 32) has 17 bits: exact, as one multiply-add too)
        s[0] = __builtin_fmaf(d, ubyte(w[9 + (j & 1)], j >> 1), -32.0f * d);
    }
};

// the 6-bit scales and minima of a super-block's 8 groups (scale_min_k) as bytes: s[0..1], m[0..1]
__device__ __forceinline__ void k_scales(uint32_t *h) {
    const uint32_t a = h[0], b = h[1], c = h[2];
    h[0] = a & 0x3F3F3F3Fu;
    h[1] = (c & 0x0F0F0F0Fu) | ((a >> 2) & 0x30303030u);
    h[2] = b & 0x3F3F3F3Fu;
    h[3] = ((c >> 4) & 0x0F0F0F0Fu) | ((b >> 2) & 0x30303030u);
}

template <> struct MX<QT_Q4_K> {
    static constexpr int NW = 13, MAP = HALVES;
    static constexpr bool MIN = true, SUB = false, CHAIN = false, DEN = true;
    static constexpr int SHIFT = 4;  // codes() takes code << SHIFT
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
        ld16(R.b0 + (128 * u + 16 * q), w);
        ld16(R.b0 + (128 * u + 64 + 16 * q), w + 4);
        ld16(R.b1 + 16 * u, w + 8);
    }
    __device__ static void arrange(uint32_t *w) {
        quarter_exchange(w);
        quarter_exchange(w + 4);
        k_scales(w + 9);
    }
    __device__ static v4u frag(const uint32_t *w, int j, int, const uint8_t *) {
        const int i = 2 * (j >> 1), sh = j & 1 ? 0 : 4;
        return codes((w[i] << sh) & 0xF0F0F0F0u, (w[i + 1] << sh) & 0xF0F0F0F0u);
    }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *m) {
        s[0] = ubyte(w[9 + (j >> 2)], j & 3);
        m[0] = ubyte(w[11 + (j >> 2)], j & 3);
    }
    __device__ static void super(const uint32_t *w, float &d, float &dm) { d = h2f(w[8]), dm = h2f(w[8] >> 16); }
};

template <> struct MX<QT_Q5_K> {
    static constexpr int NW = 15, MAP = HALVES;
    static constexpr bool MIN = true, SUB = false, CHAIN = false, DEN = true;
    static constexpr int SHIFT = 3;  // codes() takes code << SHIFT
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
        ld16(R.b0 + (128 * u + 16 * q), w);
        ld16(R.b0 + (128 * u + 64 + 16 * q), w + 4);
        w[8] = *reinterpret_cast<const uint32_t *>(R.b1 + (32 * u + 4 * q));
        w[9] = *reinterpret_cast<const uint32_t *>(R.b1 + (32 * u + 16 + 4 * q));
        ld16(R.b2 + 16 * u, w + 10);
    }
    __device__ static void arrange(uint32_t *w) {
        quarter_exchange(w);
        quarter_exchange(w + 4);
        k_scales(w + 11);
    }
    __device__ static v4u frag(const uint32_t *w, int j, int, const uint8_t *) {
        const int i = 2 * (j >> 1);
        const uint32_t rot = (uint32_t) (j + 25) & 31u;  // bit 8k + j to 8k + 7
        const uint32_t h0 = __builtin_amdgcn_alignbit(w[8], w[8], rot), h1 = __builtin_amdgcn_alignbit(w[9], w[9], rot);
        const uint32_t l0 = j & 1 ? w[i] >> 1 : w[i] << 3, l1 = j & 1 ? w[i + 1] >> 1 : w[i + 1] << 3;
        return codes((h0 & 0x80808080u) | (l0 & 0x78787878u), (h1 & 0x80808080u) | (l1 & 0x78787878u));
    }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *m) {
        s[0] = ubyte(w[11 + (j >> 2)], j & 3);
        m[0] = ubyte(w[13 + (j >> 2)], j & 3);
    }
    __device__ static void super(const uint32_t *w, float &d, float &dm) { d = h2f(w[10]), dm = h2f(w[10] >> 16); }
};

// (codes 0 .. 63 with the minimum 32 s, as the vector kernels take it)
template <> struct MX<QT_Q6_K> {
    static constexpr int NW = 17, MAP = HALVES;
    static constexpr bool MIN = true, SUB = true, CHAIN = false, DEN = true;
    static constexpr int SHIFT = 2;  // codes() takes code << SHIFT
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
        ld16(R.b0 + (128 * u + 16 * q), w);
        ld16(R.b0 + (128 * u + 64 + 16 * q), w + 4);
        ld16(R.b1 + (64 * u + 16 * q), w + 8);
        const U16p t = *reinterpret_cast<const U16p *>(R.b2 + 18 * u);  // (2-byte aligned)
        w[12] = t.w[0], w[13] = t.w[1], w[14] = t.w[2], w[15] = t.w[3];
        w[16] = ld2(R.b2 + (18 * u + 16));
    }
    __device__ static void arrange(uint32_t *w) {
        quarter_exchange(w);
        quarter_exchange(w + 4);
        quarter_exchange(w + 8);
    }
    __device__ static v4u frag(const uint32_t *w, int j, int, const uint8_t *) {
        const int n = j >> 2, qu = j & 3, i = 4 * n + 2 * (qu & 1);
        const uint32_t rot = (uint32_t) (2 * qu + 26) & 31u;  // bits 8k + 2qu, + 1 to 8k + 6, 7
        const uint32_t h0 = __builtin_amdgcn_alignbit(w[8 + 2 * n], w[8 + 2 * n], rot);
        const uint32_t h1 = __builtin_amdgcn_alignbit(w[9 + 2 * n], w[9 + 2 * n], rot);
        const uint32_t l0 = qu & 2 ? w[i] >> 2 : w[i] << 2, l1 = qu & 2 ? w[i + 1] >> 2 : w[i + 1] << 2;
        return codes((h0 & 0xC0C0C0C0u) | (l0 & 0x3C3C3C3Cu), (h1 & 0xC0C0C0C0u) | (l1 & 0x3C3C3C3Cu));
    }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *m) {
        const int n = j >> 2, qu = j & 3, b = 8 * n + 2 * qu;
        m[0] = s[0] = sbyte(w[12 + (b >> 2)], b & 3);
        m[1] = s[1] = sbyte(w[12 + (b >> 2)], (b & 3) + 1);
    }
    __device__ static void super(const uint32_t *w, float &d, float &dm) { d = h2f(w[16]), dm = 32.0f * d; }
};

// IQ3_S: the codebook as bf16 magnitudes (4 a point, 8 bytes) and the sign bytes as masks of 8 bf16 (16 bytes), in LDS
__device__ __forceinline__ void iq3s_tab_load(int tid, int nth, uint32_t (&g)[2]) {  // nth >= 256
    g[0] = kIq3sGrid[tid & 511];
    g[1] = kIq3sGrid[(tid + nth) & 511];
}
__device__ __forceinline__ void iq3s_tab_fill(uint8_t *tab, int tid, int nth, const uint32_t (&gs)[2]) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int i = tid + k * nth;
        if (i >= 512) break;
        const uint32_t g = gs[k];
        *reinterpret_cast<v2u *>(tab + 8 * i) =
            v2u{pack_f((float) (g & 0xFFu), (float) ((g >> 8) & 0xFFu)), pack_f((float) ((g >> 16) & 0xFFu), (float) (g >> 24))};
    }
    for (uint32_t i = tid; i < 256; i += nth) {
        v4u m;
#pragma unroll
        for (int k = 0; k < 4; ++k) m[k] = ((i >> (2 * k)) & 1u) << 15 | ((i >> (2 * k + 1)) & 1u) << 31;
        *reinterpret_cast<v4u *>(tab + 4096 + 16 * i) = m;
    }
}

template <> struct MX<QT_IQ3_S> {
    static constexpr int NW = 16, MAP = GRID;
    static constexpr bool MIN = false, SUB = false, CHAIN = false, DEN = false;
    template <class R_> __device__ static void load(const R_ &R, int u, int q, uint32_t *w) {
        ld16(R.b0 + (64 * u + 16 * q), w);
        struct __attribute__((packed, aligned(4))) A4 { uint32_t w[4]; };
        const A4 s0 = *reinterpret_cast<const A4 *>(R.b1 + (44 * u + 8)), s1 = *reinterpret_cast<const A4 *>(R.b1 + (44 * u + 24));
#pragma unroll
        for (int k = 0; k < 4; ++k) w[4 + k] = s0.w[k], w[8 + k] = s1.w[k];
        w[12] = *reinterpret_cast<const uint32_t *>(R.b1 + 44 * u);
        w[13] = *reinterpret_cast<const uint32_t *>(R.b1 + (44 * u + 4));
        w[14] = *reinterpret_cast<const uint32_t *>(R.b1 + (44 * u + 40));
        w[15] = ld2(R.b2 + 2 * u);
    }
    // after the exchange word j holds, by quarter, the two words of group 2j and the two of group 2j + 1; frag() wants
    // quarters 0, 2 on the group's first word and 1, 3 on its second
    __device__ static void arrange(uint32_t *w) { quarter_exchange(w); }
    __device__ static v4u frag(const uint32_t *w, int j, int lane, const uint8_t *tab) {
        const float2 t = swap32(__uint_as_float(w[j >> 1]));
        const uint32_t g = __float_as_uint(j & 1 ? t.y : t.x);
        const uint32_t q = (uint32_t) lane >> 4, p = (q & 1u) << 1 | q >> 1;  // the lane's run of 8 values
        const uint32_t c = g >> (16 * (q >> 1));
        const uint32_t h = (w[12 + (j >> 2)] >> (8 * (j & 3))) >> (2 * p);
        const v2u a = *reinterpret_cast<const v2u *>(tab + 8 * ((c & 255u) | (h & 1u) << 8));
        const v2u b = *reinterpret_cast<const v2u *>(tab + 8 * (((c >> 8) & 255u) | (h & 2u) << 7));
        const v4u m = *reinterpret_cast<const v4u *>(tab + 4096 + 16 * ((w[4 + j] >> (8 * p)) & 255u));
        return v4u{a.x ^ m.x, a.y ^ m.y, b.x ^ m.z, b.y ^ m.w};
    }
    __device__ static void scale(const uint32_t *w, int j, float *s, float *) {
        const float d = h2f(w[15]);  // (exact as one multiply-add: 16 bits)
        s[0] = __builtin_fmaf(2.0f * d, ubyte((w[14] >> (4 * (j & 1))) & 0x0F0F0F0Fu, j >> 1), d);
    }
};

template <uint32_t TY> constexpr int mx_tab_bytes() {
    return iq4_fmt<TY>() ? 32768 : (TY == QT_IQ3_S ? 8192 : 0);
}
template <uint32_t TY> __device__ __forceinline__ void mx_tab_load(int tid, int nth, uint32_t (&g)[2]) {
    if constexpr (TY == QT_IQ3_S) iq3s_tab_load(tid, nth, g);
}
template <uint32_t TY> __device__ __forceinline__ void mx_tab_fill(uint8_t *tab, int tid, int nth, const uint32_t (&g)[2]) {
    if constexpr (iq4_fmt<TY>()) iq4_pairs_fill(tab, tid, nth);
    else if constexpr (TY == QT_IQ3_S) iq3s_tab_fill(tab, tid, nth, g);
}

// LDS of a workgroup of W waves: the format's table, a piece a wave for the x split (64 fragments of 8 values x 3 parts,
// the group sums, the exponents), two buffers of 16 waves' partial sums
constexpr int MX_X = 64 * 48, MX_GRP = 4 * 48;
// (the sums of x of a token tile: 4 tokens x 8 groups, twice that for SUB; the formats without a minimum leave them out)
constexpr int mx_sums(bool min, bool sub) { return min ? (sub ? 256 : 128) : 0; }
// Whether the second of a wave's two units keeps its split x in LDS, where every tile reads it again: where the 128 VGPRs of
// a workgroup of 1024 threads do not hold two units of x, their words and the sums of x.  In registers Q5_K and Q6_K
// spilled 41 and 34 (20000 x 8192, one token, 46.2 / 46.5 us; so 30.5 / 33.6); where two fit, LDS is slower (IQ4_XS 2560 x
// 8192 8.0 / 8.4 us, and 9.6 instead of 8.3 for two tokens).
template <uint32_t TY> constexpr bool mx_stay(int upw, int maxt) {
    return upw == 2 && maxt == 1024 && MX<TY>::MIN && MX<TY>::NW >= 15;
}
template <uint32_t TY> constexpr int mx_wave(int upw, int ntile, int maxt) {  // (STAY: a piece for each of the two rounds)
    return (mx_stay<TY>(upw, maxt) ? 2 : 1) * MX_X + 64 + upw * ntile * mx_sums(MX<TY>::MIN, MX<TY>::SUB);
}
template <uint32_t TY> constexpr int mx_lds(int W, int upw, int ntile, int maxt) {
    return mx_tab_bytes<TY>() + W * mx_wave<TY>(upw, ntile, maxt) + 2 * 16 * ntile * 256;
}

// x = hi + mid + lo, each in the high 16 bits of a float: exact from |x| = 2^-110 on, where lo's low bits are zero by
// construction.  Below, bf16 ends (its smallest value is 2^-133) and lo's low bits are what it does not hold.  An
// infinity or NaN is all in hi.
__device__ __forceinline__ void split3(float x, uint32_t &h, uint32_t &m, uint32_t &l) {
    x = __builtin_canonicalizef(x);  // (a quiet NaN stays one without its low bits; folded into the product x comes from)
    h = __float_as_uint(x) & 0xFFFF0000u;
    float r = x - __uint_as_float(h);
    r = __builtin_amdgcn_fmed3f(r, r, 0.0f);  // (r; 0 where r is a NaN, of an infinity or a NaN)
    m = __float_as_uint(r) & 0xFFFF0000u;
    l = __float_as_uint(r - __uint_as_float(m));
}

// N values (4 or 8) in pairs
template <int N> __device__ __forceinline__ void split_n(const float *v, uint32_t *h, uint32_t *m, uint32_t *l) {
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
        uint32_t h0, m0, l0, h1, m1, l1;
        split3(v[2 * k], h0, m0, l0);
        split3(v[2 * k + 1], h1, m1, l1);
        h[k] = pack_hi(h0, h1), m[k] = pack_hi(m0, m1), l[k] = pack_hi(l0, l1);
    }
}

// Formats that split a single token's x over all lanes (MxX::split1): those without sums of x and a scale, for which the
// second path costs registers past 80 (Q6_K 6144 x 2560 8.7 / 10.7 us with it, IQ4_XS 512 x 2560 4.52 / 4.41).
template <uint32_t TY> constexpr bool mx_one(int ntile) { return ntile == 1 && !MX<TY>::DEN && !MX<TY>::MIN; }

// One unit of x of tokens t0 .. t0 + 3 (indices past nt - 1 repeat it; their results are not stored): load() requests
// it, split() makes the wave's A operands of it.  f[j] is lane (m, q)'s operand of group j: row m = token m / 4, part
// m % 4 (the unused fourth row reads lo again).  Two tokens a round through the wave's LDS, 8 values a lane.
//   sums (MIN), in the LDS: [token][group] of x (SUB: [token][group][half]);
//   The scale of x, a power of two.  DEN: x is scaled by 2^xexp, of the unit's largest.  Else a token's slice of x (the
//   wave's one or two units) is scaled by 2^MX_UP where all of it is below 2^-63 (up: the lanes of such tokens, by round),
//   so that values too small for an exact split (split3) have one.  A slice with a larger value is not scaled: what it may
//   lose is below 2^-133, 2^-70 of that value.  No sum overflows by it: scaled values are below 2^-10, less than 1 / 512
//   (the values of two units) beside any weight.  On an x of size 1e-36: 5e-5 off 64 bits unscaled, 1e-7 scaled.
//   Scaled under a branch instead, or split a second time where bits are lost, it cost 30 registers.
constexpr int MX_UP = 53;
template <uint32_t TY> struct MxX {
    static constexpr int MAP = MX<TY>::MAP, NS = MX<TY>::SUB ? 2 : 1;
    static constexpr bool MIN = MX<TY>::MIN, DEN = MX<TY>::DEN;
    f4v a[2], b[2];
    __device__ __forceinline__ void load(const float *__restrict__ x, int cols, int u, int t0, int nt, int lane, bool single) {
        const int q = lane & 3, gl = (lane >> 2) & 7, ts = lane >> 5;
        const int p = MAP == GRID ? (q & 1) << 1 | q >> 1 : q;
        constexpr bool RUNS = MAP == RUN || MAP == GRID;
        const int o0 = 256 * u + 32 * gl + (RUNS ? 8 * p : 4 * q), o1 = o0 + (RUNS ? 4 : 16);
        if (single && nt - t0 == 1) {  // one token: half of a quarter's 8 values a lane (split1)
            const float *xp = x + (size_t) t0 * cols;
            if constexpr (MAP == NIBBLES) {
                const f2v c = *reinterpret_cast<const f2v *>(xp + o0 + 2 * ts), d = *reinterpret_cast<const f2v *>(xp + o1 + 2 * ts);
                a[0] = f4v{c[0], d[0], c[1], d[1]};
            } else {
                a[0] = *reinterpret_cast<const f4v *>(xp + (ts ? o1 : o0));
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (r == 1 && nt - t0 <= 2) break;
            const float *xp = x + (size_t) min(t0 + 2 * r + ts, nt - 1) * cols;
            a[r] = *reinterpret_cast<const f4v *>(xp + o0);
            b[r] = *reinterpret_cast<const f4v *>(xp + o1);
        }
    }
    static __device__ __forceinline__ float quad(float s) {  // the sum over the four quarters: lanes xor 1, then xor 2
        s += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0xB1, 0xf, 0xf, false));
        s += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x4E, 0xf, 0xf, false));
        return s;
    }
    // x's scale: the largest magnitude (of the token's 256 values) to just under 2^120
    static __device__ __forceinline__ int scale_of(float mx) { return 246 - (int) (__float_as_uint(mx) >> 23); }
    template <int N> static __device__ __forceinline__ void scale_up(uint64_t up, float *v) {
        const float sc = __builtin_amdgcn_inverse_ballot_w64(up) ? __builtin_ldexpf(1.0f, MX_UP) : 1.0f;
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] *= sc;
    }
    static __device__ __forceinline__ void fence() {
        // (LDS operations of a wave are done in order; the fences keep the compiler to it)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // where a lane's operand of group 0 is after a split() of that many rounds that stays in LDS
    static __device__ __forceinline__ int piece(int rounds, int lane) {
        const int row = lane & 15, tk = row >> 2, part = min(row & 3, 2);
        return (rounds > 1 ? (tk >> 1) * MX_X : 0) + ((tk & 1) * 32 + (lane >> 4)) * 48 + 16 * part;
    }
    // split() of one token, the same bits with half the work a lane (mx_one)
    __device__ __forceinline__ void split1(int lane, uint8_t *lds, v4u *f, const uint64_t *up) const {
        const int q = lane & 3, gl = (lane >> 2) & 7, ts = lane >> 5;
        float v[4] = {a[0][0], a[0][1], a[0][2], a[0][3]};
        uint32_t h[2], m[2], l[2];
        scale_up<4>(up[0], v);
        split_n<4>(v, h, m, l);
        v2u *dst = reinterpret_cast<v2u *>(lds + (gl * 4 + q) * 48 + 8 * ts);
        dst[0] = v2u{h[0], h[1]};
        dst[2] = v2u{m[0], m[1]};
        dst[4] = v2u{l[0], l[1]};
        fence();
        const uint8_t *src = lds + (lane >> 4) * 48 + 16 * min(lane & 3, 2);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = *reinterpret_cast<const v4u *>(src + j * MX_GRP);
        fence();
    }
    __device__ __forceinline__ void split(bool stay, int rounds, int lane, uint8_t *lds, v4u *f, int *exps, float *sums, const uint64_t *up,
                                          int &xexp) const {
        const int q = lane & 3, gl = (lane >> 2) & 7, ts = lane >> 5;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (r >= rounds) break;
            float v[8];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[MAP == NIBBLES ? 2 * k : k] = a[r][k];
                v[MAP == NIBBLES ? 2 * k + 1 : 4 + k] = b[r][k];
            }
            if constexpr (MIN) {
                float s0 = (v[0] + v[1]) + (v[2] + v[3]), s1 = (v[4] + v[5]) + (v[6] + v[7]);
                if constexpr (NS == 2) s0 = quad(s0), s1 = quad(s1);
                else s0 = quad(s0 + s1);
                if (q == 0) {
                    float *to = sums + ((2 * r + ts) * 8 + gl) * NS;
                    to[0] = s0;
                    if constexpr (NS == 2) to[1] = s1;
                }
            }
            if constexpr (DEN) {
                float mx = 0.0f;  // (NaNs are passed over)
#pragma unroll
                for (int k = 0; k < 8; ++k) mx = fmaxf(mx, fabsf(v[k]));
                mx = row_max(mx);
                mx = fmaxf(mx, swz_xor16(mx));  // over the token's 256 values
                const int e = scale_of(mx);
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = ldexpf(v[k], e);
                if ((lane & 31) == 0) exps[ts] = e;
            } else {
                scale_up<8>(up[r], v);
            }
            uint32_t h[4], m[4], l[4];
            split_n<8>(v, h, m, l);
            v4u *dst = reinterpret_cast<v4u *>(lds + (stay ? r * MX_X : 0) + ((ts * 8 + gl) * 4 + q) * 48);
            dst[0] = v4u{h[0], h[1], h[2], h[3]}, dst[1] = v4u{m[0], m[1], m[2], m[3]}, dst[2] = v4u{l[0], l[1], l[2], l[3]};
            fence();
            const int row = lane & 15, tk = row >> 2, part = min(row & 3, 2);
            if (!stay && (r == 0 || (tk >> 1) == 1)) {
                const uint8_t *src = lds + (((tk & 1) * 8) * 4 + (lane >> 4)) * 48 + 16 * part;
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] = *reinterpret_cast<const v4u *>(src + j * MX_GRP);
            }
            if constexpr (DEN)
                if (r == 0 || (lane >> 5) == 1) xexp = exps[(lane >> 4) & 1];
            fence();
        }
    }
};

__device__ __forceinline__ f4v mx_mma(const v4u &a, const v4u &b, const f4v &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f4v mx_mma16(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, v2u{a0, a1}),
                                                     __builtin_bit_cast(s16x4, v2u{b0, b1}), f4v{0.0f, 0.0f, 0.0f, 0.0f}, 0,
                                                     0, 0);
}
__device__ __forceinline__ float mx_sum3(const f4v &d) { return d[0] + (d[1] + d[2]); }

// one unit's products (lane (r, c): weight row r, token c of each token tile); the groups' sums in two chains
// fx(i, j): the operand of token tile i, group j
template <uint32_t TY, int NTILE, class FX>
__device__ __forceinline__ void mx_unit(uint32_t *w, const FX &fx, const float *sums,
                                        const int (&xexp)[NTILE], int lane, const uint8_t *tab, float *out) {
    using F = MX<TY>;
    const f4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float acc[NTILE][2], mins[NTILE][2];
#pragma unroll
    for (int i = 0; i < NTILE; ++i) acc[i][0] = acc[i][1] = mins[i][0] = mins[i][1] = 0.0f;
    F::arrange(w);
    constexpr int NS = MxX<TY>::NS;
    f4v xs[NTILE][2 * NS];  // the sums of token lane / 16, by group
    if constexpr (F::MIN) {
#pragma unroll
        for (int i = 0; i < NTILE; ++i)
#pragma unroll
            for (int k = 0; k < 2 * NS; ++k)
                xs[i][k] = *reinterpret_cast<const f4v *>(sums + (i * 4 + (lane >> 4)) * 8 * NS + 4 * k);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const v4u b = F::frag(w, j, lane, tab);
        float s[2], m[2];
        F::scale(w, j, s, m);
#pragma unroll
        for (int i = 0; i < NTILE; ++i) {
            float &a = acc[i][j & 1], &n = mins[i][j & 1];
            const v4u f = fx(i, j);
            if constexpr (F::SUB) {
                const f4v d0 = mx_mma16(f.x, f.y, b.x, b.y), d1 = mx_mma16(f.z, f.w, b.z, b.w);
                a = __builtin_fmaf(s[0], mx_sum3(d0), a);
                a = __builtin_fmaf(s[1], mx_sum3(d1), a);
                n = __builtin_fmaf(m[0], xs[i][j >> 1][2 * j & 3], n);
                n = __builtin_fmaf(m[1], xs[i][j >> 1][(2 * j + 1) & 3], n);
            } else {
                const f4v d = mx_mma(f, b, zero);
                if constexpr (F::CHAIN) {
                    // (a weight is a bf16 value: where it is infinite or NaN the product is hi's, while mid and lo,
                    // often zero, give NaN)
                    a += __builtin_isfinite(d[0]) ? mx_sum3(d) : d[0];
                } else {
                    a = __builtin_fmaf(s[0], mx_sum3(d), a);
                    if constexpr (F::MIN) n = __builtin_fmaf(m[0], xs[i][j >> 2][j & 3], n);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NTILE; ++i) {
        float v = acc[i][0] + acc[i][1];
        if constexpr (F::MIN) {
            float d, dm;
            F::super(w, d, dm);
            // (the power of two last: before d, a sum near fp32's smallest values would lose bits that d v has)
            v = __builtin_fmaf(-dm, mins[i][0] + mins[i][1], ldexpf(d * v, 133 - F::SHIFT - xexp[i]));
        }
        out[i] += v;
    }
}

// One weight's tiles blk, blk + nblk, ... for tokens t0 .. t0 + 4 NTILE - 1 (of nt).  W = waves of the workgroup, U =
// units of a row; wave w sums units w UPW ..
template <uint32_t TY, int NTILE, int UPW, int MAXT>
__device__ __forceinline__ void mx_walk(const PP &P, int rows, int rt, int U, const float *__restrict__ x, int cols, int t0, int nt,
                                        float *__restrict__ y, int blk, int nblk, uint8_t *lds) {
    using F = MX<TY>;
    constexpr bool HALF = TY == QT_BF16, STAY = mx_stay<TY>(UPW, MAXT);
    const int tid = threadIdx.x, lane = tid & 63, W = blockDim.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *tab = lds;
    constexpr int WAVE = mx_wave<TY>(UPW, NTILE, MAXT), SUMS = mx_sums(F::MIN, F::SUB) / 4;  // (SUMS: floats)
    uint8_t *mine = lds + mx_tab_bytes<TY>() + wv * WAVE;
    int *exps = reinterpret_cast<int *>(mine + (STAY ? 2 : 1) * MX_X);
    float *sums = reinterpret_cast<float *>(exps + 16);
    float *red = reinterpret_cast<float *>(lds + mx_tab_bytes<TY>() + W * WAVE);
    const int r16 = lane & 15, q = lane >> 4, ntiles = (rows + rt - 1) / rt;
    const int u0 = wv * UPW;
    const bool two = UPW == 1 || u0 + 1 < U;  // (UPW = 2) the last wave may have one unit only
    const auto load = [&](int tile, int k, uint32_t *w, bool first = true, bool second = true) {
        const RP32 R = row_planes32(P, min(tile * rt + min(r16, rt - 1), rows - 1));
        if (first) F::load(R, min(u0 + k, U - 1), q, w);
        if constexpr (HALF)
            if (second) F::load2(R, min(u0 + k, U - 1), q, w);
        __builtin_amdgcn_sched_barrier(0);  // (requested here, not where the words are first used)
    };
    // The table's points (IQ3_S), x, then the first tile's words are requested before the first wait (a second unit's words
    // and half of a BF16 unit's after x is split: no registers before).  The points first, so that the table is written
    // while the rest is on its way: loads come back in order, and behind the words the table waited for them (IQ3_S 640 x
    // 2560, 1 / 8 tokens, 5.3 / 7.4 -> 5.1 / 7.0 us; two units a wave have no registers for it).
    uint32_t points[2];
    if constexpr (UPW == 1) mx_tab_load<TY>(tid, blockDim.x, points);
    MxX<TY> xr[UPW][NTILE];
#pragma unroll
    for (int k = 0; k < UPW; ++k)
#pragma unroll
        for (int i = 0; i < NTILE; ++i) xr[k][i].load(x, cols, min(u0 + k, U - 1), t0 + 4 * i, nt, lane, mx_one<TY>(NTILE));
    __builtin_amdgcn_sched_barrier(0);
    // One buffer of a unit's words, requested again as soon as its products have read it (UPW = 2: one for each of the
    // wave's units).  Two buffers, the next tile's words requested before the first products, were slower everywhere:
    // 10.0 against 8.9 us for IQ4_XS 10240 x 2560 at one token, 38.1 against 35.4 us for 100000 x 2560; the tiles of the
    // CU's other workgroup hide the latency.
    uint32_t wa[F::NW], wb[UPW == 2 ? F::NW : 1];
    const int n = blk < ntiles ? (ntiles - 1 - blk) / nblk + 1 : 0;  // the workgroup's tiles blk + i nblk
    const auto tile = [&](int i) { return blk + i * nblk; };
    load(blk, 0, wa, true, false);
    if constexpr (UPW == 2) mx_tab_load<TY>(tid, blockDim.x, points);
    mx_tab_fill<TY>(tab, tid, blockDim.x, points);
    v4u f[STAY ? 1 : UPW][NTILE][8];
    int xexp[UPW][NTILE];
    uint64_t up[NTILE][2] = {}, down[NTILE] = {};  // the lanes of scaled tokens: of x, by round, and of the results
    const bool one = mx_one<TY>(NTILE) && nt - t0 == 1;
    const auto rounds = [&](int i) { return nt - t0 - 4 * i > 2 ? 2 : 1; };
    if constexpr (!F::DEN) {
        // A value of at least 2^-63 has its exponent's first or second bit set (an infinity or a NaN too).  First one value a
        // lane, of all tokens at once: a lane of each half with no smaller one settles it (all values of every unit and
        // round, looked at before its split, cost 0.1 to 0.2 us at 8 tokens: BF16 96 x 2560 4.86 unscaled / 5.07 / 4.80 so).
        const auto large = [&](int i, int r, bool all) {
            uint32_t m = 0;
#pragma unroll
            for (int k = 0; k < UPW; ++k) {
                const f4v &a = xr[k][i].a[r], &b = xr[k][i].b[r];
                m |= __float_as_uint(a[0]);
                if (!all) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) m |= __float_as_uint(a[e]) | (one ? 0u : __float_as_uint(b[e]));
            }
            return m & 0x60000000u;
        };
        uint32_t least = ~0u;
#pragma unroll
        for (int i = 0; i < NTILE; ++i) {
            least = min(least, large(i, 0, false));
            if (rounds(i) > 1) least = min(least, large(i, 1, false));
        }
        const uint64_t some = __ballot(least != 0);
        if (one ? some == 0 : (uint32_t) some == 0 || (some >> 32) == 0)
#pragma unroll
            for (int i = 0; i < NTILE; ++i)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    if (r >= rounds(i)) break;
                    const uint64_t big = __ballot(large(i, r, true) != 0);
                    const uint64_t b0 = one ? big : (uint32_t) big, b1 = one ? big : big >> 32;
                    up[i][r] = (b0 ? 0 : 0xFFFFFFFFull) | (b1 ? 0 : 0xFFFFFFFFull << 32);
                    down[i] |= ((up[i][r] & 0xFFFF) | ((up[i][r] >> 32) & 0xFFFF) << 16) << (32 * r);
                }
    }
#pragma unroll
    for (int k = 0; k < UPW; ++k)
#pragma unroll
        for (int i = 0; i < NTILE; ++i) {
            float *s = sums + (k * NTILE + i) * SUMS;
            const bool stay = STAY && k > 0;
            v4u *to = f[stay ? 0 : k][i];
            if (one) xr[k][i].split1(lane, mine, to, up[i]);
            else xr[k][i].split(stay, rounds(i), lane, mine, to, exps, s, up[i], xexp[k][i]);
        }
    if constexpr (HALF) load(blk, 0, wa, false, true);
    if constexpr (UPW == 2) load(blk, 1, wb);
    const uint8_t *f1 = mine + MxX<TY>::piece(rounds(0), lane);  // STAY (UPW = 2, NTILE = 1)
    if constexpr (mx_tab_bytes<TY>() > 0) lds_barrier();
    int it = 0;
    float acc[NTILE];
    const auto products = [&](int k, uint32_t *w) {
        float *s = sums + k * NTILE * SUMS;
        if (STAY && k > 0)
            mx_unit<TY, NTILE>(w, [&](int, int j) { return *reinterpret_cast<const v4u *>(f1 + j * MX_GRP); }, s, xexp[k], lane, tab, acc);
        else
            mx_unit<TY, NTILE>(w, [&](int i, int j) { return f[STAY ? 0 : k][i][j]; }, s, xexp[k], lane, tab, acc);
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < NTILE; ++i) acc[i] = 0.0f;
    };
    const auto finish = [&](int tile) {
        float *buf = red + (it & 1) * (16 * NTILE * 64);
#pragma unroll
        for (int i = 0; i < NTILE; ++i) {
            if constexpr (!F::DEN) acc[i] *= __builtin_amdgcn_inverse_ballot_w64(down[i]) ? __builtin_ldexpf(1.0f, -MX_UP) : 1.0f;
            buf[(wv * NTILE + i) * 64 + lane] = acc[i];
        }
        lds_barrier();  // (the buffers alternate: this one is written again only after the next tile's barrier)
        // one wave a token tile (in turn) sums the waves' words, a token at a time: lane (r, g) those of waves g, g + 4,
        // g + 8, g + 12 of row r (room for 16 is there; those past the last wave are read and left out), then the four
        // lanes of a row meet by lane swaps
#pragma unroll
        for (int i = 0; i < NTILE; ++i)
            if (wv == (it * NTILE + i) % W) {
                const int row = tile * rt + r16;
                for (int c = 0; c < 4 && t0 + 4 * i + c < nt; ++c) {
                    float v[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[k] = buf[((q + 4 * k) * NTILE + i) * 64 + 16 * c + r16];
#pragma unroll
                    for (int k = 1; k < 4; ++k) v[k] = q + 4 * k < W ? v[k] : 0.0f;  // (W >= 4)
                    float s = add_xor32((v[0] + v[1]) + (v[2] + v[3]));
                    const float2 o = swap16(s);
                    s = o.x + o.y;
                    if (lane < rt && row < rows) y[(size_t) (t0 + 4 * i + c) * rows + row] = s;
                }
            }
        ++it;
    };
    const auto whole = [&](int i, uint32_t *w) {
        clear();
        products(0, w);
        finish(tile(i));
    };
    // Every pass of a loop requests the same words, and it ends at its test alone: a pass that requests fewer would make
    // the compiler's waits take nothing newer to be in flight.  The last tiles come after it.
    int i = 0;
    if constexpr (UPW == 2) {
        for (; i + 1 < n; ++i) {
            clear();
            products(0, wa);
            load(tile(i + 1), 0, wa);
            if (two) products(1, wb);
            load(tile(i + 1), 1, wb);
            finish(tile(i));
        }
        if (i < n) {
            clear();
            products(0, wa);
            if (two) products(1, wb);
            finish(tile(i));
        }
    } else {
        for (; i + 1 < n; ++i) {
            clear();
            products(0, wa);
            load(tile(i + 1), 0, wa);
            finish(tile(i));
        }
        if (i < n) whole(i, wa);
    }
}

// MAXT: the most threads of the workgroup (768: 168 VGPRs a lane, 1024: 128).  Six waves a SIMD (80 VGPRs) where x takes 32
// registers: the 10 waves of a 2560-column tile go 3, 3, 2, 2 to the SIMDs, so that two workgroups a CU need room for six
// (at 81 VGPRs, five a SIMD, the second one waited: Q5_K 8192 x 2560 10.4 instead of 8.7 us).
constexpr int mx_waves(int ntile, int upw, int maxt) { return ntile == 1 && upw == 1 && maxt == 768 ? 6 : 1; }
template <uint32_t TY, int NTILE, int UPW, int MAXT>
__global__ void __launch_bounds__(MAXT, mx_waves(NTILE, UPW, MAXT)) k_gemv_mx(PP P, int rows, int rt, int U, const float *__restrict__ x, int cols, int nt,
                                                  float *__restrict__ y) {
    extern __shared__ float4 xs[];
    mx_walk<TY, NTILE, UPW, MAXT>(P, rows, rt, U, x, cols, 4 * NTILE * blockIdx.y, nt, y, blockIdx.x, gridDim.x,
                            reinterpret_cast<uint8_t *>(xs));
}

template <int NTILE, int MAXT, int I, int N, uint32_t TY, uint32_t... R>
__device__ __forceinline__ void mx_grp_walk(const GParts<N> &ps, int blk, int U, const float *__restrict__ x, int cols,
                                            int nt, uint8_t *lds) {
    if (blk < ps.p[I].nwg) mx_walk<TY, NTILE, 1, MAXT>(ps.p[I].P, ps.p[I].rows, ps.p[I].rt, U, x, cols, 0, nt, ps.p[I].out, blk, ps.p[I].nwg, lds);
    else if constexpr (sizeof...(R) > 0) mx_grp_walk<NTILE, MAXT, I + 1, N, R...>(ps, blk - ps.p[I].nwg, U, x, cols, nt, lds);
}
// several weights over one x: workgroups [0, nwg_0) walk part 0, the next nwg_1 part 1, and so on
template <int NTILE, int MAXT, uint32_t... TS>
__global__ void __launch_bounds__(MAXT, mx_waves(NTILE, 1, MAXT)) k_gemv_mx_grp(GParts<sizeof...(TS)> ps, int U, const float *__restrict__ x, int cols,
                                                      int nt) {
    extern __shared__ float4 xs[];
    mx_grp_walk<NTILE, MAXT, 0, sizeof...(TS), TS...>(ps, blockIdx.x, U, x, cols, nt, reinterpret_cast<uint8_t *>(xs));
}

// workgroups of W waves and lds bytes that a CU holds (queried once per kernel and W)
template <typename K> int mx_per_cu(K kern, int *cache, int W, int lds, int &out) {
    if (!cache[W]) {
        int n = 0;
        FN_CK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, 64 * W, (size_t) lds));
        cache[W] = std::max(1, n);
    }
    out = cache[W];
    return 0;
}

// Rows of a tile: 16, or 8 or 4 for a weight of fewer than 128 tiles, so that more CUs stream it (a lane past a short
// tile's rows repeats the last one, whose result it does not store).  One token, us, 16 rows a tile against this: BF16
// 96 x 2560 5.32 / 4.29, 640 x 2560 5.82 / 4.60, IQ4_XS 512 x 2560 4.79 / 4.72.  At 256 tiles instead of 128, 2560 x 6144
// (160 tiles of 16) would take tiles of 8, 320 on 256 CUs: 8.7 / 11.3.
inline int mx_tile_rows(int rows) {
    int rt = 16;
    while (rt > 4 && (rows + rt - 1) / rt < 128) rt /= 2;
    return rt;
}

template <uint32_t TY, int NTILE, int UPW, int MAXT>
int mx_launch(const QLayout &L, const uint8_t *packed, const float *x, int nt, float *y, hipStream_t st) {
    static int cache[17] = {};
    const int U = L.cols / 256, W = (U + UPW - 1) / UPW, lds = mx_lds<TY>(W, UPW, NTILE, MAXT), rt = mx_tile_rows(L.rows);
    const int halves = (nt + 4 * NTILE - 1) / (4 * NTILE), ntiles = (L.rows + rt - 1) / rt;
    int per_cu = 0;
    if (mx_per_cu(k_gemv_mx<TY, NTILE, UPW, MAXT>, cache, W, lds, per_cu)) return -1;
    if (g_ov_wpc) per_cu = std::max(1, g_ov_wpc / W);
    const int nwg = g_persist ? std::min(ntiles, std::max(1, device_cus() * per_cu / halves)) : ntiles;
    hipLaunchKernelGGL((k_gemv_mx<TY, NTILE, UPW, MAXT>), dim3((unsigned) nwg, (unsigned) halves), dim3(64 * W), (size_t) lds,
                       st, planes(L, packed), L.rows, rt, U, x, L.cols, nt, y);
    FN_CK(hipGetLastError());
    return 0;
}

template <uint32_t TY>
int mx_gemv_t(const QLayout &L, const uint8_t *packed, const float *x, int nt, float *y, hipStream_t st) {
    const int U = L.cols / 256;
    if constexpr (TY != QT_BF16) {
        if (U > 24) return mx_launch<TY, 1, 2, 1024>(L, packed, x, nt, y, st);
        if (U > 16) return mx_launch<TY, 1, 2, 768>(L, packed, x, nt, y, st);
    }
    if (U > 12)
        return nt > 4 ? mx_launch<TY, 2, 1, 1024>(L, packed, x, nt, y, st) : mx_launch<TY, 1, 1, 1024>(L, packed, x, nt, y, st);
    return nt > 4 ? mx_launch<TY, 2, 1, 768>(L, packed, x, nt, y, st) : mx_launch<TY, 1, 1, 768>(L, packed, x, nt, y, st);
}

template <int NTILE, int MAXT, uint32_t... TS>
int mx_grp_launch(const QLayout *const *L, const PP *P, float *const *y, const float *x, int nt, hipStream_t st) {
    constexpr int N = sizeof...(TS);
    static int cache[17] = {};
    const int U = L[0]->cols / 256, W = U, lds = std::max({mx_lds<TS>(W, 1, NTILE, MAXT)...});
    int per_cu = 0;
    if (mx_per_cu(k_gemv_mx_grp<NTILE, MAXT, TS...>, cache, W, lds, per_cu)) return -1;
    // Tiles are of one size for all parts.  `walk`, the most tiles that a workgroup takes, is the fewest for which the
    // workgroups are resident at once.  Where a CU holds two, the ones left over are shared out by tiles: the walk alone
    // would leave some CUs two workgroups and others one (DeltaNet set, one token: 16.6 us so, 11.7 shared out); where it
    // holds one, more of them only split x more often (8 tokens: 16.0 us by the walk, 18.3 shared out).
    // `walk` is of the part with the lightest rows; the others walk fewer tiles, by their bytes: a CU streams a BF16 tile
    // (128 KB at 4096 columns) in the time of three or four of IQ4_XS, and one workgroup with four of them was what the
    // launch waited for (attention set, one token, in equal tiles / by bytes: 2560 columns 11.9 / 9.9 us, 4096 columns
    // 19.3 / 12.2, where the vector kernels take 15.4; 8 tokens 15.9 / 12.3 and 21.2 / 15.2).
    const int budget = device_cus() * per_cu;
    GParts<N> ps;
    int tiles[N], w[N], all = 0, rows = 0, walk = 0, nwg = 0;
    size_t light = L[0]->row_bytes;
    for (int i = 1; i < N; ++i) light = std::min(light, L[i]->row_bytes);
    for (int i = 0; i < N; ++i) rows += L[i]->rows;
    const int rt = mx_tile_rows(rows);
    for (int i = 0; i < N; ++i) all += tiles[i] = (L[i]->rows + rt - 1) / rt;
    do {
        ++walk, nwg = 0;
        for (int i = 0; i < N; ++i) {
            const int k = std::max(1, (int) (walk * light / L[i]->row_bytes));
            nwg += w[i] = (tiles[i] + k - 1) / k;
        }
    } while (nwg > budget && nwg > N);
    // (a part of a few tiles, such as the 96 rows of alpha and beta, has a workgroup for each)
    nwg = 0;
    for (int i = 0; i < N; ++i) nwg += w[i] = tiles[i] <= 8 ? tiles[i] : w[i];
    const int left = per_cu > 1 ? std::max(0, std::min(budget, all) - nwg) : 0;
    nwg = 0;
    for (int i = 0; i < N; ++i) {
        w[i] = std::min(tiles[i], w[i] + (int) ((long long) left * tiles[i] / all));
        ps.p[i] = GPart{P[i], L[i]->rows, w[i], y[i], rt};
        nwg += w[i];
    }
    hipLaunchKernelGGL((k_gemv_mx_grp<NTILE, MAXT, TS...>), dim3((unsigned) nwg), dim3(64 * W), (size_t) lds, st, ps, U, x,
                       L[0]->cols, nt);
    FN_CK(hipGetLastError());
    return 0;
}
template <uint32_t... TS>
int mx_grp(const QLayout *const *L, const PP *P, float *const *y, const float *x, int nt, hipStream_t st) {
    if (L[0]->cols > 12 * 256)
        return nt > 4 ? mx_grp_launch<2, 1024, TS...>(L, P, y, x, nt, st) : mx_grp_launch<1, 1024, TS...>(L, P, y, x, nt, st);
    return nt > 4 ? mx_grp_launch<2, 768, TS...>(L, P, y, x, nt, st) : mx_grp_launch<1, 768, TS...>(L, P, y, x, nt, st);
}

}  // namespace
}  // namespace fn
