// Quantized matmul on the f16 matrix cores for the weight types the int8
// digit kernels do not take (Q8_0, Q4_0, Q4_1, Q5_0, Q5_1; Q2K, Q3K, Q5K),
// from a few rows up to prefill sizes.
//
// Exactness.  Every level of these formats times its integer sub-block scale
// and every 8-bit activation level is a whole number that f16 holds exactly,
// and their products are exact.  The sum of one block is below 2^24 (Q8_0
// 5.2e5, Q2K 1.5e6, Q3K 4.2e6) and so exact in the f32 accumulator: the matrix
// core returns the same integer block dot the reference forms (k_quants.rs:
// 287-304, 419-440, 513-544, 677-691, 899-948, 1071-1152, 1524-1605), as a float
// and without a conversion.  Q5K's can reach 63 x 31 x 128 x 256 = 6.4e7, see there.
//
// Scales.  The 32-element types scale every 32 K: y += (d_w d_a) I.  Both
// scales are f16, so their outer product over a 32 x 32 tile is one more
// MFMA with a single non-zero K slot, exact in f32, and the epilogue is one
// fma per output element (with the product formed on the vector units it is
// two, and with an int8 contraction three).  The K types scale every 256 K:
// y += d_a (d_w I1 - dmin I2), where I2 = sum_g m_g bsum_g is one K = 16 MFMA
// of the sub-block mins by the 16 block sums, exact for the same reason.
//
// Q5K.  On activations of one sign I1 passes 2^24, and d_w I1 and dmin I2 are
// several times their difference.  The levels are therefore expanded less 16,
// which keeps the running sum small, and one more MFMA adds
// sum_g (16 sc_g - kappa m_g) bsum_g with kappa = dmin / d_w rounded to a whole number
// of 0 .. 31, so that the larger part of the cancellation is between whole numbers
// (below 2^24 unless a whole block's levels are extreme); what the min term then
// still has is dmin - kappa d_w.  Relative L2 error against 64 bits on rows of 10 + 0.3 N(0, 1),
// matvec / with levels 0 .. 31 / this: K = 256 1.48e-7 / 2.62e-7 / 3.8e-8, 4096
// 1.60e-7 / 2.73e-7 / 4.7e-8; on N(0, 1) rows 4096 1.04e-7 / 6.2e-8 / 4.8e-8.
//
// Operands.  Weight columns are MFMA operand A (expanded to f16 in registers
// right before use: a nibble or byte b becomes 0x6400 | b = 1024 + b, then one
// packed add or fma), activation rows operand B, read as f16 in MFMA order
// from the activation image (H16Img).  Lane (column or row l & 31, half
// l >> 5) holds elements 16 half .. 16 half + 15 of each 32-element chunk, as
// two K = 16 steps.
//
// Summation.  Long chains of f32 additions are split so that the rounding
// error stays at or below that of the matvec kernels' lane tree: four blocks,
// then four stages, then the rest; super-blocks in eights.  Wavefronts that
// split K, and the stores of a long K, are added in 64 bits.
#include <type_traits>

#include "xnq_device.h"
#include "xnq_internal.h"

namespace xnq {

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kThreads = 512, kWaves = 8;

// What one 32-column stage of a weight type is: CH chunks of 32 K, SEG bytes
// of the q plane per column, fetched with LDS DMA as P pieces of PB bytes (16
// where blocks are 8-byte aligned, else 4) in NI instructions of a wavefront,
// column after column.  The scales of the plane types (Q8_0, Q4_0) take one
// more instruction.
template <int DT>
struct HT {
    static constexpr bool kK = is_kquant(DT);
    static constexpr int kCH = kK ? 8 : 4;
    static constexpr int kSeg = DT == XNQ_Q8_0 ? 128 : DT == XNQ_Q4_0 ? 64 : kK ? (int)raw_stride(DT) : 4 * (int)raw_stride(DT);
    static constexpr int kPB = DT == XNQ_Q2K || DT == XNQ_Q4_1 ? 4 : 16;
    static constexpr int kP = kSeg / kPB;
    static constexpr int kNI = (32 * kP + 63) / 64;
    static constexpr bool kPlaneD = DT == XNQ_Q8_0 || DT == XNQ_Q4_0;  // d in a plane of its own
    static constexpr bool kMin32 = DT == XNQ_Q4_1 || DT == XNQ_Q5_1;
    static constexpr bool kMinK = DT == XNQ_Q2K || DT == XNQ_Q5K;
    static constexpr int kSlot = kNI * 64 * kPB + (kPlaneD ? 256 : 0);  // one stage in LDS
    static constexpr int kND = kNI + (kPlaneD ? 1 : 0);                 // DMA instructions of a stage
    static constexpr int kDl = kK ? 256 : 0;  // d_w, dmin by column (K types)
};

// LDS offset of piece p of column c in a stage.  Powers of two are swizzled so
// that the eight lanes of one read phase fall in different banks; the odd and
// 6-piece strides spread by themselves.
template <int DT>
__device__ __forceinline__ uint32_t piece_off(uint32_t c, uint32_t p) {
    if (DT == XNQ_Q8_0) return (c * 8 + (p ^ ((c >> 1) & 7))) * 16;
    if (DT == XNQ_Q4_0) return (c * 4 + (p ^ ((c >> 2) & 3))) * 16;
    return (c * HT<DT>::kP + p) * HT<DT>::kPB;
}

// 1024 + byte for bytes (0, 1) and (2, 3) of x
__device__ __forceinline__ h2 magic01(uint32_t x) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u));
}
__device__ __forceinline__ h2 magic23(uint32_t x) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u));
}
// 256 + byte / 4 for bytes (0, 1) and (2, 3) of x
__device__ __forceinline__ h2 quarter01(uint32_t x) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x5c5c5c5cu, x, 0x04010400u));
}
__device__ __forceinline__ h2 quarter23(uint32_t x) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x5c5c5c5cu, x, 0x04030402u));
}
__device__ __forceinline__ h2 splat2(float v) {
    const _Float16 h = (_Float16)v;
    return h2{h, h};
}

// Per-lane plane offsets of the DMA of a 32-column tile, without the stage's
// own offset.
template <int DT>
struct WOff {
    uint32_t row[HT<DT>::kNI], in[HT<DT>::kNI];  // column's row offset, offset in the stage's segment
    uint32_t d;
};

template <int DT>
__device__ __forceinline__ void weight_offsets(WOff<DT>& o, const WView& w, uint32_t col0, uint32_t lane) {
    using T = HT<DT>;
#pragma unroll
    for (int i = 0; i < T::kNI; i++) {
        const uint32_t idx = min(i * 64 + lane, 32u * T::kP - 1), c = idx / T::kP;
        uint32_t p = idx % T::kP;
        if (DT == XNQ_Q8_0) p ^= (c >> 1) & 7;
        if (DT == XNQ_Q4_0) p ^= (c >> 2) & 3;
        o.row[i] = min(col0 + c, w.n - 1) * w.q_row;
        o.in[i] = p * T::kPB;
    }
    o.d = T::kPlaneD ? min(col0 + (lane >> 1), w.n - 1) * w.d_row + (lane & 1) * 4 : 0u;
}

// DMA of stage st into the LDS slot at byte address `to`.  A stage past the end of the row
// (K not a multiple of 128) re-reads the row's last piece; its scales are zeroed, as are the
// activation's for those chunks in the image (an infinite one would make them NaN).
template <int DT, bool DV>
__device__ __forceinline__ void issue_weights(const WOff<DT>& o, const WView& w, uint32_t st, uint32_t to) {
    using T = HT<DT>;
#pragma unroll
    for (int i = 0; i < T::kNI; i++) {
        uint32_t off = st * T::kSeg + o.in[i];
        if (!T::kK && !(T::kPlaneD && DV)) off = min(off, w.q_row - T::kPB);
        if (T::kPB == 16) dma16(w.q, o.row[i] + off, to + i * 1024);
        else dma4(w.q, o.row[i] + off, to + i * 256);
    }
    if (T::kPlaneD && DV) dma4(w.d, o.d + st * 8, to + T::kNI * 1024);
}

// 16 bytes of LDS at a 4-byte aligned address
__device__ __forceinline__ uint4 lds16(const uint8_t* p) {
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
    return make_uint4(q[0], q[1], q[2], q[3]);
}

// bits 0-3 of t, one to bit 4 of each byte (t < 16: the product has no carries)
__device__ __forceinline__ uint32_t spread_bit4(uint32_t t) { return (__umul24(t, 0x00204081u) & 0x01010101u) << 4; }

// The bytes of chunk j that a lane expands: its 16 levels' low bits, and high
// bits where the type has them apart.
struct Bytes {
    uint4 v, w;
};

// `slot` is the stage in LDS, c the column, h the lane half.
template <int DT>
__device__ __forceinline__ void read_chunk(Bytes& r, const uint8_t* slot, uint32_t c, int j, uint32_t h) {
    const uint8_t* col = slot + c * HT<DT>::kSeg;  // (block types)
    if constexpr (DT == XNQ_Q8_0) {
        r.v = *reinterpret_cast<const uint4*>(slot + piece_off<DT>(c, 2 * j + h));
    } else if constexpr (DT == XNQ_Q4_0) {
        r.v = *reinterpret_cast<const uint4*>(slot + piece_off<DT>(c, j));
    } else if constexpr (DT == XNQ_Q4_1) {
        r.v = lds16(col + j * 20 + 4);
    } else if constexpr (DT == XNQ_Q5_0 || DT == XNQ_Q5_1) {
        r.v = lds16(col + j * 24 + 8);
        r.w.x = *reinterpret_cast<const uint32_t*>(col + j * 24 + 4);
    } else if constexpr (DT == XNQ_Q5K) {
        // chunk j = 2i + s: nibble s of qs bytes 32i .. 32i+31, fifth bit j of qh
        r.v = *reinterpret_cast<const uint4*>(col + 48 + 32 * (j >> 1) + 16 * h);
        r.w = *reinterpret_cast<const uint4*>(col + 16 + 16 * h);
    } else {
        // Q2K, Q3K: chunk j = 4h' + t: bits 2t of qs bytes 32h' .. 32h'+31; Q3K's third bit j of hmask
        r.v = lds16(col + (DT == XNQ_Q2K ? 16 : 32) + 32 * (j >> 2) + 16 * h);
        if (DT == XNQ_Q3K) r.w = lds16(col + 16 * h);
    }
}

// What a stage needs of its weights beside the levels.
template <int DT>
struct Scales {
    uint4 hd;                            // K types: the block header's words
    uint2 d[HT<DT>::kK ? 1 : 4];      // 32-element types: operand of the scale product, chunk j
    uint2 m[HT<DT>::kMin32 ? 4 : 1];  // and of the min product
    uint4 mn;                            // K types: min-term operand
    uint4 rest;                          // Q5K: 16 sc - kappa m, laid out like it,
    float bias;                          // and -272, or -256 where d_w is not finite
};

// Operand A of chunk j: the lane's 16 levels (times the sub-block scale, K
// types) as two K = 16 steps.
template <int DT>
__device__ __forceinline__ void expand(const Bytes& r, int j, uint32_t h, const Scales<DT>& S, h8* a) {
    const uint4& hd = S.hd;
    const uint32_t v[4] = {r.v.x, r.v.y, r.v.z, r.v.w}, w[4] = {r.w.x, r.w.y, r.w.z, r.w.w};
    uint32_t x[4];  // four levels a dword, as bytes
    float bias = 0.f, sc = 0.f;
    if constexpr (DT == XNQ_Q8_0) {
#pragma unroll
        for (int d = 0; d < 4; d++) x[d] = v[d] ^ 0x80808080u;
        bias = -1152.f;
    } else if constexpr (!HT<DT>::kK) {
#pragma unroll
        for (int d = 0; d < 4; d++) {
            x[d] = (v[d] >> (4 * h)) & 0x0F0F0F0Fu;
            if (DT == XNQ_Q5_0 || DT == XNQ_Q5_1) x[d] |= spread_bit4((w[0] >> (16 * h + 4 * d)) & 15u);
        }
        bias = DT == XNQ_Q4_0 ? -1032.f : DT == XNQ_Q5_0 ? -1040.f : -1024.f;
    } else if constexpr (DT == XNQ_Q5K) {
#pragma unroll
        for (int d = 0; d < 4; d++)  // four times the level
            x[d] = ((j & 1 ? v[d] >> 2 : v[d] << 2) & 0x3C3C3C3Cu) | ((j > 6 ? w[d] >> 1 : w[d] << (6 - j)) & 0x40404040u);
        const Q4KScales q = q4k_scales(hd.y, hd.z, hd.w);
        sc = (float)(((j < 4 ? q.sc_lo : q.sc_hi) >> (8 * (j & 3))) & 0xffu);
    } else {
#pragma unroll
        for (int d = 0; d < 4; d++) x[d] = (v[d] >> (2 * (j & 3))) & 0x03030303u;
        if constexpr (DT == XNQ_Q3K) {  // the lane's 16 elements are sub-block 2j + h
#pragma unroll
            for (int d = 0; d < 4; d++) x[d] |= (j >= 2 ? w[d] >> (j - 2) : w[d] << (2 - j)) & 0x04040404u;
            sc = (float)(q3k_scale(hd.x, hd.y, hd.z, (int)(2 * j + h)) - 32);
        } else {
            const uint32_t hw = (j >> 1) == 0 ? hd.x : (j >> 1) == 1 ? hd.y : (j >> 1) == 2 ? hd.z : hd.w;
            sc = (float)((hw >> (8 * (2 * (j & 1) + h))) & 15u);
        }
    }
    h2 q[8];
#pragma unroll
    for (int d = 0; d < 4; d++) {
        q[2 * d] = DT == XNQ_Q5K ? quarter01(x[d]) : magic01(x[d]);
        q[2 * d + 1] = DT == XNQ_Q5K ? quarter23(x[d]) : magic23(x[d]);
    }
    if constexpr (!HT<DT>::kK) {
        const h2 b = splat2(bias);
#pragma unroll
        for (int d = 0; d < 8; d++) q[d] = q[d] + b;
    } else if constexpr (DT == XNQ_Q3K) {
        const h2 b = splat2(-1028.f), s = splat2(sc);
#pragma unroll
        for (int d = 0; d < 8; d++) q[d] = (q[d] + b) * s;
    } else {
        // Q2K (1024 + q) sc - 1024 sc, Q5K (256 + q) sc - 272 sc = (q - 16) sc, exact: 1024 sc
        // is a 4-bit number times 2^10, 272 sc = 17 sc <= 1071 times 2^4
        const h2 s = splat2(sc), b = splat2((DT == XNQ_Q5K ? S.bias : -1024.f) * sc);
#pragma unroll
        for (int d = 0; d < 8; d++) q[d] = __builtin_elementwise_fma(q[d], s, b);
    }
    a[0] = h8{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y};
    a[1] = h8{q[4].x, q[4].y, q[5].x, q[5].y, q[6].x, q[6].y, q[7].x, q[7].y};
}

__device__ __forceinline__ f16v mfma16(h8 a, h8 b, f16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// the K = 8 step takes half the operand registers: for the rank-1 products
__device__ __forceinline__ f16v mfma8(uint2 a, uint2 b) {
    return __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(h4, a), __builtin_bit_cast(h4, b), f16v{}, 0, 0, 0);
}
__device__ __forceinline__ h8 as_h8(uint4 v) { return __builtin_bit_cast(h8, v); }

// An infinite activation scale (an infinity in the block) makes every block dot of the
// reference NaN: a zero sum times it, or main and min terms of one sign.  (The
// quantizer does the same for the f16 image.)  So does an infinite weight scale of Q3K,
// whose reference multiplies eight sums of either sign by it (k_quants.rs:1071-1152).
__device__ __forceinline__ float finite_or_nan(float d) { return fmaf(d, 0.0f, d); }

// Reads a stage's scales from its slot; K types also leave d_w and dmin by
// column at dl (a wavefront's own LDS: its operations stay in order).
template <int DT, bool DV>
__device__ __forceinline__ void read_scales(Scales<DT>& S, const WView& w, const uint8_t* slot, uint8_t* dl,
                                            uint32_t col0, uint32_t lane, uint32_t st, uint32_t nch) {
    using T = HT<DT>;
    const uint32_t c = lane & 31, h = lane >> 5;
    const uint8_t* col = slot + c * T::kSeg;
    if constexpr (T::kK) {
        uint32_t dd;
        if constexpr (DT == XNQ_Q5K) {
            S.hd = *reinterpret_cast<const uint4*>(col);
            dd = S.hd.x;
        } else if constexpr (DT == XNQ_Q2K) {
            S.hd = lds16(col);  // the 16 scale / min bytes
            dd = *reinterpret_cast<const uint32_t*>(col + 80);
        } else {
            S.hd = lds16(col + 96);
            dd = S.hd.w & 0xffffu;
        }
        if constexpr (DT == XNQ_Q5K) {  // (the rest: read_rest)
            const float dw = f16_bits_to_f32(dd & 0xffffu);
            S.bias = dw - dw == 0.f ? -272.f : -256.f;
        } else {
            // [dw 32][dmin 32] (Q3K: d_w twice)
            const float d = f16_bits_to_f32(T::kMinK && h ? dd >> 16 : dd & 0xffffu);
            reinterpret_cast<float*>(dl)[lane] = DT == XNQ_Q3K ? finite_or_nan(d) : d;
        }
        if constexpr (DT == XNQ_Q2K) {
            // mins of sub-blocks (16 elements each) 8h .. 8h + 7
            h8 mv;
            const uint32_t b0 = h ? S.hd.z : S.hd.x, b1 = h ? S.hd.w : S.hd.y;
#pragma unroll
            for (int t = 0; t < 8; t++) mv[t] = (_Float16)(float)(((t < 4 ? b0 : b1) >> (8 * (t & 3) + 4)) & 15u);
            S.mn = __builtin_bit_cast(uint4, mv);
        }
    } else {
        uint32_t dv[4];
        if constexpr (T::kPlaneD && DV) {
            const uint2 v = *reinterpret_cast<const uint2*>(slot + T::kNI * 1024 + c * 8);
            dv[0] = v.x & 0xffffu; dv[1] = v.x >> 16; dv[2] = v.y & 0xffffu; dv[3] = v.y >> 16;
        } else if constexpr (T::kPlaneD) {
            const uint16_t* dp = reinterpret_cast<const uint16_t*>(w.d + min(col0 + c, w.n - 1) * w.d_row);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t v = dp[min(st * 4 + j, nch - 1)];
                dv[j] = st * 4 + j < nch ? v : 0u;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t f = *reinterpret_cast<const uint32_t*>(col + j * (int)raw_stride(DT));
                const bool live = st * 4 + j < nch;
                dv[j] = live ? f & 0xffffu : 0u;
                if constexpr (T::kMin32) S.m[j] = make_uint2(live && h == 0 ? f >> 16 : 0u, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) S.d[j] = make_uint2(h == 0 ? dv[j] : 0u, 0);
    }
}

// Operand B of chunk j's min product out of a stage's four f16 sums: the other
// three stay out of it also where the weight operand is zero, since a sum that
// overflowed f16 (a block's sum past 65504, its scale still finite) would make
// them 0 x inf = NaN.
__device__ __forceinline__ uint2 chunk_sum(const uint2& s, int j) {
    const uint32_t v = j < 2 ? s.x : s.y;
    return make_uint2(j & 1 ? v >> 16 : v & 0xffffu, 0);
}

// One 32 x 32 unit (a chunk of a 32-element type by a row tile): the matrix
// products, and their fold into the running sum t.
template <int DT>
struct Unit {
    f16v I, sc, p;
};
template <int DT>
__device__ __forceinline__ void unit_mma(Unit<DT>& u, const h8* a, const Scales<DT>& S, int j, const uint4* b,
                                         const uint2& bd, const uint2& bs) {
    u.I = mfma16(a[0], as_h8(b[0]), f16v{});
    u.sc = mfma8(S.d[j], bd);
    u.I = mfma16(a[1], as_h8(b[1]), u.I);
    if constexpr (HT<DT>::kMin32) u.p = mfma8(S.m[j], bs);
}
template <int DT>
__device__ __forceinline__ void unit_add(const Unit<DT>& u, bool first, f16v& t) {
#pragma unroll
    for (int e = 0; e < 16; e++) {
        if constexpr (HT<DT>::kMin32) {
            // per block, as the reference's vec_dot: the min and main terms cancel
            const float v = fmaf(u.I[e], u.sc[e], u.p[e]);
            t[e] = first ? v : t[e] + v;
        } else {
            t[e] = first ? u.I[e] * u.sc[e] : fmaf(u.I[e], u.sc[e], t[e]);
        }
    }
}

// Each byte of w (<= 63) times f (1 or 16) as two f16 whole numbers.
__device__ __forceinline__ void bytes_twice(uint32_t w, float f, h2* r) {
#pragma unroll
    for (int t = 0; t < 4; t++) {  // (1024 + byte) f - 1024 f
        const h2 v = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u + 0x00010001u * t));
        r[t] = __builtin_elementwise_fma(v, splat2(f), splat2(-1024.f * f));
    }
}

// Q5K: the operands of the block sums, and at dl d_w and what kappa d_w leaves of dmin.
// Apart from read_scales: nothing needs them before the super-block's products are done.
template <int DT>
__device__ __forceinline__ void read_rest(Scales<DT>& S, uint8_t* dl, uint32_t lane) {
    const uint32_t h = lane >> 5;
    const Q4KScales q = q4k_scales(S.hd.y, S.hd.z, S.hd.w);
    const float dw = f16_bits_to_f32(S.hd.x & 0xffffu), dm = f16_bits_to_f32(S.hd.x >> 16);
    const bool ok = dw - dw == 0.f;
    // (any whole number would be right: an infinite or NaN quotient is clamped, d_w's own
    // infinity or NaN meets the sums as they are)
    const float kappa = ok ? rintf(fminf(fmaxf(dm * __builtin_amdgcn_rcpf(dw), 0.f), 31.f)) : 0.f;
    h2 m[4], c[4];
    bytes_twice(h ? q.m_hi : q.m_lo, 1.f, m);
    bytes_twice(h ? q.sc_hi : q.sc_lo, ok ? 16.f : 0.f, c);
#pragma unroll
    for (int t = 0; t < 4; t++) c[t] = __builtin_elementwise_fma(m[t], splat2(-kappa), c[t]);  // |.| <= 1953
    S.mn = __builtin_bit_cast(uint4, h8{m[0].x, m[0].y, m[1].x, m[1].y, m[2].x, m[2].y, m[3].x, m[3].y});
    S.rest = __builtin_bit_cast(uint4, h8{c[0].x, c[0].y, c[1].x, c[1].y, c[2].x, c[2].y, c[3].x, c[3].y});
    reinterpret_cast<float*>(dl)[lane] = h == 0 ? dw : ok ? fmaf(-kappa, dw, dm) : dm;
}

// A super-block's sums I (and the min sums) of a 32 x 32 tile into the output.
template <int DT>
__device__ __forceinline__ void super_unit(f16v I, const Scales<DT>& S, const uint4& bs, float da, const float* dw,
                                           const float* dm, f16v& out) {
    if constexpr (DT == XNQ_Q5K) I = mfma16(as_h8(S.rest), as_h8(bs), I);
    if constexpr (HT<DT>::kMinK) {
        const f16v I2 = mfma16(as_h8(S.mn), as_h8(bs), f16v{});
#pragma unroll
        for (int e = 0; e < 16; e++) out[e] = fmaf(da, fmaf(dw[e], I[e], -(dm[e] * I2[e])), out[e]);
    } else {
#pragma unroll
        for (int e = 0; e < 16; e++) out[e] = fmaf(da * dw[e], I[e], out[e]);
    }
}

// ---------------------------------------------------------------------------
// Few rows, or few tiles: a workgroup owns 32 weight columns and 32 TM rows,
// and its eight wavefronts split K, so that a weight of a few thousand columns
// still puts two wavefronts on every SIMD.  Each wavefront streams its share of
// the weights through its own LDS ring (LDS DMA in whole cache lines) and its
// share of the activation image straight into registers (a stage ahead); there
// is no barrier until the eight partial tiles are added through LDS.
//
// The ring holds two stages beyond the present one, but the DMA does not run that
// far ahead: a stage's is issued after the activation loads of the next one, and the
// waits that the compiler places for those loads know nothing of it and so drain it
// too, for the most part within the stage it was issued in (with one row tile Q5K's
// all of it).  A stage therefore still meets the latency of its weights in part.
// ---------------------------------------------------------------------------
// The eight wavefronts' partials of four outputs, added in 64 bits: one rounding
// for the eight, which pays for those of the longer chains over a wavefront's
// stages (relative L2 error against exact sums, the matvec kernels' / these, Q8_0: K = 1024
// 6.6e-8 / 4.7e-8, 4096 7.4e-8 / 6.3e-8, 14336 8.4e-8 / 7.4e-8).
__device__ __forceinline__ float4 sum_waves(const float4* p, int stride) {
    double x = 0, y = 0, z = 0, w = 0;
#pragma unroll
    for (int v = 0; v < kWaves; v++) {
        const float4 q = p[v * stride];
        x += q.x;
        y += q.y;
        z += q.z;
        w += q.w;
    }
    return make_float4((float)x, (float)y, (float)z, (float)w);
}

// Operand B out of the int8 row images (ActImg) instead of the f16 image, for callers
// that hold a quantized activation of their own: the same values, at a conversion
// beside each product and loads of 16 bytes a row (all of a stage's at once, so
// that a line is used whole, was no better: Q8_0 4096 -> 1024 m = 125 21 against
// 20 us, Q5K 4096 -> 6144 m = 37 28 / 21, Q4_0 4096 -> 14336 m = 512 425 / 453).
__device__ __forceinline__ void row_quants(const uint4& v, uint4* b) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    const h2 c = splat2(-1152.f);  // 1024 + (byte + 128)
    h2 q[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        q[2 * i] = magic01(d[i] ^ 0x80808080u) + c;
        q[2 * i + 1] = magic23(d[i] ^ 0x80808080u) + c;
    }
    b[0] = __builtin_bit_cast(uint4, h8{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y});
    b[1] = __builtin_bit_cast(uint4, h8{q[4].x, q[4].y, q[5].x, q[5].y, q[6].x, q[6].y, q[7].x, q[7].y});
}
__device__ __forceinline__ uint4 row_bsums(const uint4& v) {
    typedef short s8 __attribute__((ext_vector_type(8)));
    const s8 t = __builtin_bit_cast(s8, v);
    h8 h;
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = (_Float16)t[i];  // |bsum| <= 2048: exact
    return __builtin_bit_cast(uint4, h);
}

template <int DT, int TM, bool DV, bool ROWS>
__global__ __launch_bounds__(kThreads) void h16_ksplit_kernel(WView w, AView a, uint32_t m, uint32_t m_tiles,
                                                              uint32_t n_tiles, float* __restrict__ y) {
    using T = HT<DT>;
    constexpr int kU = T::kCH * TM;       // (chunk, tile) units of a stage
    // Units whose operand B is in flight: 8, but half of that for Q4_1 and Q5_1 on two row tiles,
    // whose min products' operands are registers more: with 8 they spilled 72 and 52, with 4 9
    // and 5 (8192 -> 6144 m = 64, graph steps, us, 60.6 / 33.0 and 46.6 / 32.0).
    constexpr int kPD = T::kMin32 && TM == 2 && !ROWS ? 4 : kU < 8 ? kU : 8;
    constexpr int kSlots = 3, kWaveLds = kSlots * T::kSlot + T::kDl;
    constexpr int kRed = kWaves * TM * 4 * 64 * 16;
    constexpr int kLds = kWaves * kWaveLds > kRed ? kWaves * kWaveLds : kRed;
    static_assert(kLds <= 160 * 1024, "LDS budget");
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t total = m_tiles * n_tiles, per = (total + 7) / 8;
    const uint32_t wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // one XCD: consecutive items, one column tile
    if (wi >= total) return;
    const uint32_t mt = wi % m_tiles, nt = wi / m_tiles;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col0 = nt * 32, nch = w.k / 32;
    const uint32_t nst = (nch + T::kCH - 1) / T::kCH, wst = (nst + kWaves - 1) / kWaves;
    const uint32_t s0 = min(wave * wst, nst), s1 = min(s0 + wst, nst);
    uint8_t* wl = lds + wave * kWaveLds;
    uint8_t* dl = wl + kSlots * T::kSlot;
    const uint32_t wbase = (uint32_t)(uintptr_t)lds + wave * kWaveLds;
    const H16Img& H = a.H;
    const uint32_t lrow = lane & 31, g = lane >> 5;

    // lanes of rows past m read the last row again (their outputs are dropped)
    uint32_t rt[TM], bl[TM];
    const uint8_t* row[TM];  // ROWS: the lane's row image
#pragma unroll
    for (int i = 0; i < TM; i++) {
        rt[i] = min(mt * TM + i, ROWS ? (m - 1) / 32 : H.rts - 1);
        bl[i] = g * 32 + min(lrow, m - 1 - rt[i] * 32);
        if constexpr (ROWS) row[i] = a.img + (size_t)min(rt[i] * 32 + lrow, m - 1) * a.A.row_bytes;
    }

    f16v out[TM], mid[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) out[i] = mid[i] = f16v{};

    if (s0 < s1) {
        WOff<DT> wo;
        weight_offsets<DT>(wo, w, col0, lane);
        uint4 b[kPD][ROWS ? 1 : 2];
        uint2 bd[T::kK ? 1 : kPD];  // ROWS: f32 scale, quant sum
        float da[TM];    // K types: d_a of the stage's super-block
        uint4 bs[TM];    // and min-term operand
        uint2 bs32[TM];  // Q4_1, Q5_1: min-term operand of the stage
        auto load_unit = [&](uint32_t st, int u, int slot) {
            const int j = u / TM, i = u % TM;
            const uint32_t cj = st * T::kCH + j, c = min(cj, nch - 1);
            if constexpr (ROWS) {
                b[slot][0] = *reinterpret_cast<const uint4*>(row[i] + g * (w.k / 2) + c * 16);
                if constexpr (!T::kK) {  // (no scale past the end of the row)
                    bd[slot].x = cj < nch ? *reinterpret_cast<const uint32_t*>(row[i] + a.A.d_off + c * 4) : 0u;
                    if constexpr (T::kMin32) bd[slot].y = *reinterpret_cast<const uint32_t*>(row[i] + a.A.s_off + c * 4);
                }
                return;
            }
            const uint8_t* p = a.h16 + ((size_t)rt[i] * nch + c) * 2048 + bl[i] * 16;
            b[slot][0] = *reinterpret_cast<const uint4*>(p);
            if constexpr (!ROWS) b[slot][1] = *reinterpret_cast<const uint4*>(p + 1024);
            if constexpr (!T::kK)
                bd[slot] = *reinterpret_cast<const uint2*>(a.h16 + H.d_off + ((size_t)rt[i] * nst * 4 + cj) * 512 + lane * 8);
        };
        auto load_scales = [&](uint32_t st) {
#pragma unroll
            for (int i = 0; i < TM; i++) {
                if constexpr (ROWS) {
                    if constexpr (T::kK) {
                        da[i] = reinterpret_cast<const float*>(row[i] + a.A.d_off)[st];
                        if constexpr (T::kMinK) bs[i] = *reinterpret_cast<const uint4*>(row[i] + a.A.s_off + st * 32 + g * 16);
                    }
                } else if constexpr (T::kK) {
                    da[i] = reinterpret_cast<const float*>(a.h16 + H.d_off + ((size_t)rt[i] * nst + st) * 128)[lrow];
                    if constexpr (T::kMinK)
                        bs[i] = *reinterpret_cast<const uint4*>(a.h16 + H.s_off + ((size_t)rt[i] * nst + st) * 1024 + lane * 16);
                } else if constexpr (T::kMin32) {
                    bs32[i] = *reinterpret_cast<const uint2*>(a.h16 + H.s_off + ((size_t)rt[i] * nst + st) * 512 + lane * 8);
                }
            }
        };
        // unit u's operands, as the matrix instructions take them
        auto unit_b = [&](int u, uint4* ub) {
            if constexpr (ROWS) {
                row_quants(b[u % kPD][0], ub);
            } else {
                ub[0] = b[u % kPD][0];
                ub[1] = b[u % kPD][1];
            }
        };
        auto unit_d = [&](int u, uint2& ud, uint2& us) {
            if constexpr (ROWS) {
                const float d = __uint_as_float(bd[u % kPD].x);
                ud = make_uint2(g == 0 ? (uint32_t)f32_to_f16_bits(d) : 0u, 0);
                if constexpr (T::kMin32) {  // Q8_1's s, as the quantizer forms it
                    const float t = f16_bits_to_f32(f32_to_f16_bits((float)(int)bd[u % kPD].y));
                    us = make_uint2(g == 0 ? (uint32_t)f32_to_f16_bits(t * d) : 0u, 0);
                }
            } else {
                ud = bd[u % kPD];
                if constexpr (T::kMin32) us = chunk_sum(bs32[u % TM], u / TM);
            }
        };
        issue_weights<DT, DV>(wo, w, s0, wbase);
        issue_weights<DT, DV>(wo, w, min(s0 + 1, s1 - 1), wbase + T::kSlot);
#pragma unroll
        for (int u = 0; u < kPD; u++) load_unit(s0, u, u);
        load_scales(s0);
        asm volatile("" ::: "memory");
        issue_weights<DT, DV>(wo, w, min(s0 + 2, s1 - 1), wbase + 2 * T::kSlot);
        uint32_t slot = 0;
        for (uint32_t s = s0; s < s1; s++) {
            const uint32_t sn = min(s + 1, s1 - 1);
            // the DMA of stages s + 1 and s + 2 is younger than this stage's
            wait_vm<2 * ((T::kPlaneD && !DV) ? T::kNI : T::kND)>();
            const uint8_t* ws = wl + slot * T::kSlot;
            Scales<DT> S;
            read_scales<DT, DV>(S, w, ws, dl, col0, lane, s, nch);
            if constexpr (T::kK) {
                f16v I[TM];
#pragma unroll
                for (int j = 0; j < T::kCH; j++) {
                    if constexpr (DT == XNQ_Q5K) {
                        // (later, the two-tile form spills: 4096 -> 6144 m = 37 19.6 us against 16.8)
                        if (j == 2) read_rest<DT>(S, dl, lane);
                    }
                    h8 A[2];
                    Bytes by;
                    read_chunk<DT>(by, ws, lrow, j, g);
                    expand<DT>(by, j, g, S, A);
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        const int u = j * TM + i;
                        uint4 ub[2];
                        unit_b(u, ub);
                        I[i] = mfma16(A[0], as_h8(ub[0]), j == 0 ? f16v{} : I[i]);
                        I[i] = mfma16(A[1], as_h8(ub[1]), I[i]);
                        if (u + kPD < kU) load_unit(s, u + kPD, u % kPD);
                        else load_unit(sn, u + kPD - kU, u % kPD);
                    }
                }
                float dw[16], dm[16];
                const float* dp = reinterpret_cast<const float*>(dl) + 4 * g;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    dw[e] = dp[8 * (e >> 2) + (e & 3)];
                    if (T::kMinK) dm[e] = dp[32 + 8 * (e >> 2) + (e & 3)];
                }
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    if constexpr (ROWS)
                        super_unit<DT>(I[i], S, T::kMinK ? row_bsums(bs[i]) : uint4{}, finite_or_nan(da[i]), dw, dm, out[i]);
                    else
                        super_unit<DT>(I[i], S, bs[i], da[i], dw, dm, out[i]);
                }
            } else {
                f16v t[TM];
#pragma unroll
                for (int j = 0; j < T::kCH; j++) {
                    h8 A[2];
                    Bytes by;
                    read_chunk<DT>(by, ws, lrow, j, g);
                    expand<DT>(by, j, g, S, A);
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        const int u = j * TM + i;
                        Unit<DT> un;
                        uint4 ub[2];
                        uint2 ud, us{};
                        unit_b(u, ub);
                        unit_d(u, ud, us);
                        unit_mma<DT>(un, A, S, j, ub, ud, us);
                        unit_add<DT>(un, j == 0, t[i]);
                        if (u + kPD < kU) load_unit(s, u + kPD, u % kPD);
                        else load_unit(sn, u + kPD - kU, u % kPD);
                        // folded here: sunk to the stage's end, with the conversions in front, it spills
                        if constexpr (ROWS) asm volatile("" : "+v"(t[i]));
                    }
                }
#pragma unroll
                for (int i = 0; i < TM; i++) {
#pragma unroll
                    for (int e = 0; e < 16; e++) mid[i][e] += t[i][e];
                }
                if ((s & 3) == 3) {
#pragma unroll
                    for (int i = 0; i < TM; i++) {
#pragma unroll
                        for (int e = 0; e < 16; e++) out[i][e] += mid[i][e];
                        mid[i] = f16v{};
                    }
                }
            }
            load_scales(sn);
            // this stage's slot is read; fetch stage s + 3 into it
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue_weights<DT, DV>(wo, w, min(s + 3, s1 - 1), wbase + slot * T::kSlot);
            slot = slot == 2 ? 0 : slot + 1;
        }
        wait_vm<0>();  // no DMA may land in the reduction below
    }
    // partial tiles to LDS ([wave][tile, quad][lane] float4), then one quad of
    // one tile per wavefront, summed over the eight
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float4 v;
            v.x = out[i][4 * q] + mid[i][4 * q];
            v.y = out[i][4 * q + 1] + mid[i][4 * q + 1];
            v.z = out[i][4 * q + 2] + mid[i][4 * q + 2];
            v.w = out[i][4 * q + 3] + mid[i][4 * q + 3];
            reinterpret_cast<float4*>(lds)[(wave * (TM * 4) + i * 4 + q) * 64 + lane] = v;
        }
    __syncthreads();
    for (uint32_t iq = wave; iq < TM * 4; iq += kWaves) {
        const float4 o = sum_waves(reinterpret_cast<const float4*>(lds) + iq * 64 + lane, TM * 4 * 64);
        const uint32_t row = (mt * TM + (iq >> 2)) * 32 + lrow, n = col0 + 8 * (iq & 3) + 4 * g;
        if (row >= m) continue;
        float* yr = y + (size_t)row * w.n + n;
        if ((w.n & 3) == 0 && n + 3 < w.n) {
            *reinterpret_cast<float4*>(yr) = o;
        } else {
            if (n < w.n) yr[0] = o.x;
            if (n + 1 < w.n) yr[1] = o.y;
            if (n + 2 < w.n) yr[2] = o.z;
            if (n + 3 < w.n) yr[3] = o.w;
        }
    }
}

// ---------------------------------------------------------------------------
// The same for 16 rows, the 32-element types: a workgroup owns 32 columns and 16
// rows (the upper or lower half of a 32-row tile of the image) on 16 x 16
// tiles, where one K = 32 product is one chunk.  A wavefront's stages are a
// serial chain (activation loads, expansion, products, fold), and a workgroup
// has the CU's LDS to itself, so what counts is a stage's length: 16 rows halve
// its activation bytes and products and take a third off its vector work, and
// 32-row tiles leave CUs idle where these are still one round.  us, graph steps
// with the quantize, 32-row tiles / this, K = 4096: Q8_0 N = 1024 m = 125 14.8 /
// 13.1, N = 4096 m = 16 13.4 / 11.8 and 32 13.9 / 12.3, N = 14336 m = 16 29.1 /
// 26.3; Q4_0 N = 4096 m = 16 12.8 / 11.4; Q4_1 14.4 / 13.3; Q5_0 13.3 / 13.3 and
// Q5_1 14.5 / 14.5 (their bit planes' expansion is what counts), N = 14336
// 30.0 / 26.0.
// ---------------------------------------------------------------------------
typedef float f4v __attribute__((ext_vector_type(4)));

template <int DT>
__device__ __forceinline__ void read_chunk8(uint2& v, uint32_t& qh, const uint8_t* slot, uint32_t c, int j, uint32_t kg) {
    const uint8_t* col = slot + c * HT<DT>::kSeg;
    const uint32_t o = 8 * (kg & 1);
    if constexpr (DT == XNQ_Q8_0) {
        v = *reinterpret_cast<const uint2*>(slot + piece_off<DT>(c, 2 * j + (kg >> 1)) + o);
    } else if constexpr (DT == XNQ_Q4_0) {
        v = *reinterpret_cast<const uint2*>(slot + piece_off<DT>(c, j) + o);
    } else if constexpr (DT == XNQ_Q4_1) {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(col + j * 20 + 4 + o);
        v = make_uint2(p[0], p[1]);
    } else {
        v = *reinterpret_cast<const uint2*>(col + j * 24 + 8 + o);
        qh = *reinterpret_cast<const uint32_t*>(col + j * 24 + 4);
    }
}

// lane (column, kg = lane / 16): elements 8 kg .. 8 kg + 7 of a chunk
template <int DT>
__device__ __forceinline__ h8 expand8(const uint2& v, uint32_t qh, uint32_t kg) {
    const uint32_t d[2] = {v.x, v.y};
    h2 q[4];
    const h2 b = splat2(DT == XNQ_Q8_0 ? -1152.f : DT == XNQ_Q4_0 ? -1032.f : DT == XNQ_Q5_0 ? -1040.f : -1024.f);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        uint32_t x;
        if constexpr (DT == XNQ_Q8_0) {
            x = d[i] ^ 0x80808080u;
        } else {
            x = (d[i] >> (4 * (kg >> 1))) & 0x0F0F0F0Fu;
            if (DT == XNQ_Q5_0 || DT == XNQ_Q5_1) x |= spread_bit4((qh >> (8 * kg + 4 * i)) & 15u);
        }
        q[2 * i] = magic01(x) + b;
        q[2 * i + 1] = magic23(x) + b;
    }
    return h8{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y};
}

__device__ __forceinline__ f4v mfma16x16x32(h8 a, h8 b) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, f4v{}, 0, 0, 0);
}
__device__ __forceinline__ f4v mfma16x16x16(uint2 a, uint2 b) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, a), __builtin_bit_cast(h4, b), f4v{}, 0, 0, 0);
}

template <int DT>
__global__ __launch_bounds__(kThreads) void h16_ksplit16_kernel(WView w, AView a, uint32_t m, uint32_t m_tiles,
                                                                uint32_t n_tiles, float* __restrict__ y) {
    using T = HT<DT>;
    constexpr bool DV = true;  // the scales of planed types come with the stage (whole stages only)
    constexpr int kSlots = 3, kWaveLds = kSlots * T::kSlot;
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t total = m_tiles * n_tiles, per = (total + 7) / 8;
    const uint32_t wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // one XCD: consecutive items, one column tile
    if (wi >= total) return;
    const uint32_t mt = wi % m_tiles, nt = wi / m_tiles;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t col0 = nt * 32, nch = w.k / 32;
    const uint32_t nst = (nch + 3) / 4, wst = (nst + kWaves - 1) / kWaves;
    const uint32_t s0 = min(wave * wst, nst), s1 = min(s0 + wst, nst);
    uint8_t* wl = lds + wave * kWaveLds;
    const uint32_t wbase = (uint32_t)(uintptr_t)lds + wave * kWaveLds;
    const H16Img& H = a.H;
    const uint32_t r = lane & 15, kg = lane >> 4, rt = mt >> 1, rg = mt & 1;
    // lanes of rows past m read the last row again (their outputs are dropped)
    const uint32_t rl = min(r, m - 1 - mt * 16);
    const uint32_t b_off = (kg & 1) * 1024 + (kg >> 1) * 512 + rg * 256 + rl * 16;
    // scales and sums: the row's 8 bytes for kg == 0, else one zero entry (half 1's first)
    const uint32_t d_off = kg == 0 ? (rg * 16 + rl) * 8 : 256;

    f4v out[2], mid[2];  // the two column tiles
#pragma unroll
    for (int ct = 0; ct < 2; ct++) out[ct] = mid[ct] = f4v{};
    if (s0 < s1) {
        WOff<DT> wo;
        weight_offsets<DT>(wo, w, col0, lane);
        uint4 b[4];
        uint2 bd[4], bs = make_uint2(0, 0);
        auto load_b = [&](uint32_t st, int j) {
            const uint32_t cj = st * 4 + j, c = min(cj, nch - 1);
            b[j] = *reinterpret_cast<const uint4*>(a.h16 + ((size_t)rt * nch + c) * 2048 + b_off);
            bd[j] = *reinterpret_cast<const uint2*>(a.h16 + H.d_off + ((size_t)rt * nst * 4 + cj) * 512 + d_off);
        };
        auto load_s = [&](uint32_t st) {
            if constexpr (T::kMin32)
                bs = *reinterpret_cast<const uint2*>(a.h16 + H.s_off + ((size_t)rt * nst + st) * 512 + d_off);
        };
        issue_weights<DT, DV>(wo, w, s0, wbase);
        issue_weights<DT, DV>(wo, w, min(s0 + 1, s1 - 1), wbase + T::kSlot);
#pragma unroll
        for (int j = 0; j < 4; j++) load_b(s0, j);
        load_s(s0);
        asm volatile("" ::: "memory");
        issue_weights<DT, DV>(wo, w, min(s0 + 2, s1 - 1), wbase + 2 * T::kSlot);
        uint32_t slot = 0;
        for (uint32_t s = s0; s < s1; s++) {
            const uint32_t sn = min(s + 1, s1 - 1);
            // the DMA of stages s + 1 and s + 2 is younger than this stage's
            wait_vm<2 * T::kND>();
            const uint8_t* ws = wl + slot * T::kSlot;
            // d_w (and m) of the lane's two columns, chunks 0 .. 3: operands of the
            // rank-1 products (only lanes kg == 0 hold them)
            uint32_t dv[2][4], mv[2][4];
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                const uint32_t c = ct * 16 + r;
                if constexpr (T::kPlaneD) {
                    const uint2 v = *reinterpret_cast<const uint2*>(ws + T::kNI * 1024 + c * 8);
                    const uint32_t x = kg == 0 ? v.x : 0u, z = kg == 0 ? v.y : 0u;
                    dv[ct][0] = x & 0xffffu; dv[ct][1] = x >> 16; dv[ct][2] = z & 0xffffu; dv[ct][3] = z >> 16;
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t f = *reinterpret_cast<const uint32_t*>(ws + c * T::kSeg + j * (int)raw_stride(DT));
                        const uint32_t v = kg == 0 && s * 4 + j < nch ? f : 0u;
                        dv[ct][j] = v & 0xffffu;
                        mv[ct][j] = v >> 16;
                    }
                }
            }
            f4v t[2];
#pragma unroll
            for (int j = 0; j < 4; j++) {
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    uint2 wv;
                    uint32_t qh = 0;
                    read_chunk8<DT>(wv, qh, ws, ct * 16 + r, j, kg);
                    const f4v I = mfma16x16x32(expand8<DT>(wv, qh, kg), as_h8(b[j]));
                    const f4v sc = mfma16x16x16(make_uint2(dv[ct][j], 0), bd[j]);
                    if constexpr (T::kMin32) {
                        // per block, as the reference's vec_dot: the min and main terms cancel
                        const f4v p = mfma16x16x16(make_uint2(mv[ct][j], 0), chunk_sum(bs, j));
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float v = fmaf(I[e], sc[e], p[e]);
                            t[ct][e] = j == 0 ? v : t[ct][e] + v;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++) t[ct][e] = j == 0 ? I[e] * sc[e] : fmaf(I[e], sc[e], t[ct][e]);
                    }
                }
                load_b(sn, j);
            }
            load_s(sn);
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int e = 0; e < 4; e++) mid[ct][e] += t[ct][e];
            if ((s & 3) == 3) {
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
#pragma unroll
                    for (int e = 0; e < 4; e++) out[ct][e] += mid[ct][e];
                    mid[ct] = f4v{};
                }
            }
            // this stage's slot is read; fetch stage s + 3 into it
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue_weights<DT, DV>(wo, w, min(s + 3, s1 - 1), wbase + slot * T::kSlot);
            slot = slot == 2 ? 0 : slot + 1;
        }
        wait_vm<0>();  // no DMA may land in the reduction below
    }
    // partial tiles to LDS ([wave][column tile][lane] float4), then one column
    // tile per wavefront, summed over the eight
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < 2; ct++)
        reinterpret_cast<float4*>(lds)[(wave * 2 + ct) * 64 + lane] =
            make_float4(out[ct][0] + mid[ct][0], out[ct][1] + mid[ct][1], out[ct][2] + mid[ct][2], out[ct][3] + mid[ct][3]);
    __syncthreads();
    if (wave >= 2) return;
    const float4 o = sum_waves(reinterpret_cast<const float4*>(lds) + wave * 64 + lane, 2 * 64);
    const uint32_t row = mt * 16 + r, n = col0 + wave * 16 + 4 * kg;
    if (row >= m) return;
    float* yr = y + (size_t)row * w.n + n;
    if ((w.n & 3) == 0 && n + 3 < w.n) {
        *reinterpret_cast<float4*>(yr) = o;
    } else {
        if (n < w.n) yr[0] = o.x;
        if (n + 1 < w.n) yr[1] = o.y;
        if (n + 2 < w.n) yr[2] = o.z;
        if (n + 3 < w.n) yr[3] = o.w;
    }
}

// ---------------------------------------------------------------------------
// Prefill sizes: a workgroup owns 256 weight columns and 64 rows, K advances
// four chunks (128) a step, and the activation tile is shared through LDS.  All
// data moves by LDS DMA; one barrier per step publishes the shared pieces, and
// each wavefront waits for its own DMA by exact count.
//
// The K types: eight wavefronts; wavefront w owns columns 32w .. 32w+31 and
// every row, so each weight is expanded once per workgroup.  The activation
// tile (1 KiB pieces) goes into a three-slot ring two steps ahead, each
// wavefront's own weights (a super-block, two steps) into two slots one
// super-block ahead.
// ---------------------------------------------------------------------------
template <int DT>
struct TLay {
    using T = HT<DT>;
    static constexpr int kBSlot = 2 * 4 * 2048;
    static constexpr int kSb = 2 * 128 + (T::kMinK ? 2 * 1024 : 0);  // a super-block's d_a, sums
    static constexpr int kOffW = 3 * kBSlot;
    static constexpr int kOffSb = kOffW + kWaves * 2 * T::kSlot;
    static constexpr int kOffDl = kOffSb + 2 * kSb;
    static constexpr int kLds = kOffDl + kWaves * T::kDl;
    static_assert(kLds <= 160 * 1024, "LDS budget");
    // DMA instructions of every wavefront: per step, and per super-block
    static constexpr int kNB = 2, kNSb = 1 + (T::kMinK ? 1 : 0);
};

template <int DT>
__global__ __launch_bounds__(kThreads) void h16_super_tile_kernel(WView w, AView a, uint32_t m, uint32_t m_tiles,
                                                                  uint32_t n_tiles, float* __restrict__ y) {
    using T = HT<DT>;
    using Y = TLay<DT>;
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t total = m_tiles * n_tiles, per = (total + 7) / 8;
    const uint32_t wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // one XCD: consecutive items, which share columns
    if (wi >= total) return;
    const uint32_t mt = wi % m_tiles, nt = wi / m_tiles;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lrow = lane & 31, g = lane >> 5;
    const uint32_t col0 = nt * 256 + wave * 32, nch = w.k / 32, nsb = nch / 8, nstep = nch / 4;
    const uint32_t lbase = (uint32_t)(uintptr_t)lds;
    const H16Img& H = a.H;
    const uint32_t rt0 = mt * 2, rt1 = min(mt * 2 + 1, H.rts - 1);

    // ---- DMA: step q's activation tile, a super-block's scales and sums, its weights ----
    auto issue_b = [&](uint32_t q, uint32_t slot) {
        const uint32_t c = min(q, nstep - 1) * 4 + (wave >> 1), to = lbase + slot * Y::kBSlot + wave * 1024;
        dma16(a.h16 + ((size_t)rt0 * nch + c) * 2048 + (wave & 1) * 1024, lane * 16, to);
        dma16(a.h16 + ((size_t)rt1 * nch + c) * 2048 + (wave & 1) * 1024, lane * 16, to + 8192);
    };
    const uint8_t* const d0 = a.h16 + H.d_off + (size_t)rt0 * nsb * 128;
    auto issue_sb = [&](uint32_t sb, uint32_t slot) {
        const uint32_t sc = min(sb, nsb - 1), to = lbase + Y::kOffSb + slot * Y::kSb;
        dma4(d0 + sc * 128, (g ? (rt1 - rt0) * nsb * 128 : 0u) + lrow * 4, to);
        if constexpr (T::kMinK)  // of row tile wave & 1 (repeats are the same bytes)
            dma16(a.h16 + H.s_off + ((size_t)(wave & 1 ? rt1 : rt0) * nsb + sc) * 1024, lane * 16,
                  to + 256 + (wave & 1) * 1024);
    };
    WOff<DT> wo;
    weight_offsets<DT>(wo, w, col0, lane);
    const uint32_t wls = Y::kOffW + wave * (2 * T::kSlot);
    auto issue_w = [&](uint32_t sb, uint32_t slot) {
        issue_weights<DT, true>(wo, w, min(sb, nsb - 1), lbase + wls + slot * T::kSlot);
    };

    // two levels of sums, eight super-blocks each in the first: one chain over a long
    // K rounds off more than the matvec's lanes do
    f16v out[2], mid[2], I[2];
#pragma unroll
    for (int i = 0; i < 2; i++) out[i] = f16v{};
    issue_b(0, 0);
    issue_sb(0, 0);
    issue_w(0, 0);
    issue_b(1, 1);
    uint32_t slot = 0, free_slot = 2;
    Scales<DT> S;
    uint8_t* dl = lds + Y::kOffDl + wave * T::kDl;
    for (uint32_t sb8 = 0; sb8 < nsb; sb8 += 8) {
        const uint32_t e8 = min(sb8 + 8, nsb);
        mid[0] = mid[1] = f16v{};
        for (uint32_t sb = sb8; sb < e8; sb++) {
            const uint8_t* ws = lds + wls + (sb & 1) * T::kSlot;
            const uint8_t* sbp = lds + Y::kOffSb + (sb & 1) * Y::kSb;
#pragma unroll
            for (int p = 0; p < 2; p++) {
                // this step has landed, and every wavefront is past the previous one.  Younger
                // than its DMA: at the first step the next step's tile, at the second also the
                // next super-block's pieces
                if (p == 0) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(Y::kNB) : "memory");
                else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(Y::kNB + Y::kNSb + T::kND) : "memory");
                issue_b(2 * sb + p + 2, free_slot);
                if (p == 0) {
                    issue_sb(sb + 1, (sb + 1) & 1);
                    issue_w(sb + 1, (sb + 1) & 1);
                    read_scales<DT, true>(S, w, ws, dl, col0, lane, sb, nch);
                }
                const uint8_t* bs = lds + slot * Y::kBSlot + lane * 16;
#pragma unroll
                for (int jj = 0; jj < 4; jj++) {
                    const int j = 4 * p + jj;
                    if constexpr (DT == XNQ_Q5K) {
                        // m = 512, 4096 -> 4096, us: here 53.7, after the products 57.3, before
                        // them 59.3, with neither this nor the levels less 16 53.0
                        if (j == 7) read_rest<DT>(S, dl, lane);
                    }
                    h8 A[2];
                    Bytes by;
                    read_chunk<DT>(by, ws, lrow, j, g);
                    expand<DT>(by, j, g, S, A);
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const uint4 b0 = *reinterpret_cast<const uint4*>(bs + i * 8192 + jj * 2048);
                        const uint4 b1 = *reinterpret_cast<const uint4*>(bs + i * 8192 + jj * 2048 + 1024);
                        I[i] = mfma16(A[0], as_h8(b0), j == 0 ? f16v{} : I[i]);
                        I[i] = mfma16(A[1], as_h8(b1), I[i]);
                    }
                }
                free_slot = slot;
                slot = slot == 2 ? 0 : slot + 1;
            }
            float dw[16], dm[16];
            const float* dp = reinterpret_cast<const float*>(dl) + 4 * g;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                dw[e] = dp[8 * (e >> 2) + (e & 3)];
                if (T::kMinK) dm[e] = dp[32 + 8 * (e >> 2) + (e & 3)];
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float da = reinterpret_cast<const float*>(sbp)[i * 32 + lrow];
                uint4 ms = make_uint4(0, 0, 0, 0);
                if constexpr (T::kMinK) ms = *reinterpret_cast<const uint4*>(sbp + 256 + i * 1024 + lane * 16);
                super_unit<DT>(I[i], S, ms, da, dw, dm, mid[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) out[i][e] += mid[i][e];
    }
    wait_vm<0>();  // no DMA outlives the workgroup's LDS
    const uint32_t nb0 = col0 + 4 * g;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t row = mt * 64 + i * 32 + lrow;
        if (row >= m) continue;
        float* yr = y + (size_t)row * w.n;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t n = nb0 + 8 * q;
            if (n + 3 < w.n && (w.n & 3) == 0) {
                *reinterpret_cast<float4*>(yr + n) =
                    make_float4(out[i][4 * q], out[i][4 * q + 1], out[i][4 * q + 2], out[i][4 * q + 3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < w.n) yr[n + e] = out[i][4 * q + e];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// The 32-element types at prefill sizes.  A unit (32 x 32 x 32) is 3 MFMAs, 20
// vector operations to fold it, and 20 to 24 (Q5: 40) to expand its weights: the
// vector units bound it (issuing for 70 % of the cycles of Q4_0's dispatch, MFMAs
// for 30 %), and two wavefronts per SIMD left them idle while both waited for LDS.
// So sixteen wavefronts, four per SIMD, with one 32 x 32 tile each (a column
// group's weights are fetched once for its two wavefronts and expanded by both):
// M = 512, 4096 -> 14336, graph steps with the quantizer, weights rotated over
// 600 MB, us, 8 wavefronts of 32 x 64 on 16 x 16 tiles / this: Q4_0 153 / 136, Q8_0
// 158 / 137, Q5_0 190 / 176.  Q4_1 and Q5_1, whose min products do not fit the
// registers beside the rest, lose: 259 / 348 and 236 / 282 (part of it, Q4_1 23,
// to the shorter chains of sums below).
// Three slots of LDS where they fit, fetched two steps ahead, else two.
// ---------------------------------------------------------------------------
template <int DT>
struct BLay {
    using T = HT<DT>;
    static constexpr int kSc = 2 * 4 * 2048, kMs = kSc + 2 * 2048;  // scales, sums: offsets in a slot
    static constexpr int kBSlot = kMs + (T::kMin32 ? 2 * 512 : 0);
    static constexpr int kWSlot = 8 * T::kSlot;
    static constexpr int kSlots = 3 * (kBSlot + kWSlot) <= 160 * 1024 ? 3 : 2;
    static constexpr int kOffW = kSlots * kBSlot, kLds = kOffW + kSlots * kWSlot;
    static_assert(kLds <= 160 * 1024, "LDS budget");
};

// s_waitcnt vmcnt(n) for a wavefront-uniform n of 1 .. 8
__device__ __forceinline__ void wait_vm_n(uint32_t n) {
    switch (n) {
    case 1: wait_vm<1>(); break;
    case 2: wait_vm<2>(); break;
    case 3: wait_vm<3>(); break;
    case 4: wait_vm<4>(); break;
    case 5: wait_vm<5>(); break;
    case 6: wait_vm<6>(); break;
    case 7: wait_vm<7>(); break;
    case 8: wait_vm<8>(); break;
    default: wait_vm<0>(); break;
    }
}

template <int DT, bool DV>
__global__ __launch_bounds__(1024) void h16_block_tile_kernel(WView w, AView a, uint32_t m, uint32_t m_tiles,
                                                              uint32_t n_tiles, float* __restrict__ y) {
    using T = HT<DT>;
    using Y = BLay<DT>;
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t total = m_tiles * n_tiles, per = (total + 7) / 8;
    const uint32_t wi = (blockIdx.x & 7) * per + (blockIdx.x >> 3);  // one XCD: consecutive items, which share columns
    if (wi >= total) return;
    const uint32_t mt = wi % m_tiles, nt = wi / m_tiles;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t cw = wave & 7, rh = wave >> 3;  // column group, row tile
    const uint32_t lrow = lane & 31, g = lane >> 5;
    const uint32_t col0 = nt * 256 + cw * 32, nch = w.k / 32, nstep = (nch + 3) / 4;
    const uint32_t lbase = (uint32_t)(uintptr_t)lds;
    const H16Img& H = a.H;
    const uint32_t rt0 = mt * 2, rt1 = min(mt * 2 + 1, H.rts - 1);

    WOff<DT> wo;
    weight_offsets<DT>(wo, w, col0, lane);
    // DMA of step q: one 1 KiB piece of the activation tile per wavefront, the
    // scales from wavefronts 0 .. 3, the sums from 4, a column group's weights
    // from its two wavefronts in turn
    const uint8_t* const b0 = a.h16 + (size_t)(rh ? rt1 : rt0) * nch * 2048 + (cw & 1) * 1024;
    const uint8_t* const d0 = a.h16 + H.d_off + (size_t)(wave >> 1 ? rt1 : rt0) * nstep * 2048;
    const uint8_t* const s0 = a.h16 + H.s_off + (size_t)rt0 * nstep * 512;
    auto issue = [&](uint32_t q, uint32_t slot) {
        const uint32_t to = lbase + slot * Y::kBSlot, tw = lbase + Y::kOffW + slot * Y::kWSlot + cw * T::kSlot;
        const uint32_t qc = min(q, nstep - 1);
        dma16(b0 + (size_t)min(qc * 4 + (cw >> 1), nch - 1) * 2048, lane * 16, to + wave * 1024);
        if (wave < 4)
            dma16(d0, (qc * 4 + 2 * (wave & 1) + g) * 512 + lrow * 16, to + Y::kSc + wave * 1024);
        if (T::kMin32 && wave == 4) dma16(s0 + qc * 512, (g ? (rt1 - rt0) * nstep * 512 : 0u) + lrow * 16, to + Y::kMs);
#pragma unroll
        for (int i = 0; i < T::kNI; i++) {
            if ((i & 1) != (int)rh) continue;
            uint32_t off = qc * T::kSeg + wo.in[i];
            if (!(T::kPlaneD && DV)) off = min(off, w.q_row - T::kPB);
            if (T::kPB == 16) dma16(w.q, wo.row[i] + off, tw + i * 1024);
            else dma4(w.q, wo.row[i] + off, tw + i * 256);
        }
        if (T::kPlaneD && DV && rh == 1) dma4(w.d, wo.d + qc * 8, tw + T::kNI * 1024);
    };
    // this wavefront's DMA instructions of a step
    const uint32_t nd = 1 + (wave < 4 ? 1 : 0) + (T::kMin32 && wave == 4 ? 1 : 0) + (rh == 0 ? (T::kNI + 1) / 2 : T::kNI / 2) +
                        (T::kPlaneD && DV && rh == 1 ? 1 : 0);

    f16v out, mid;

    // The output tile, out + mid, stored (first) or added to.  Long K adds to it
    // every 16 steps: a last level of the sum that needs no registers.  It is added in
    // 64 bits, one rounding for the two sums.
    auto add3 = [](float z, float o, float t) { return (float)((double)z + (double)o + (double)t); };
    auto flush = [&](bool first) __attribute__((always_inline)) {
        uint32_t r0 = lrow;
        asm volatile("" : "+v"(r0));  // keeps the addresses out of the step loop's registers
        const uint32_t row = mt * 64 + rh * 32 + r0;
        if (row < m) {
            float* yr = y + (size_t)row * w.n;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t n = col0 + 4 * g + 8 * q;
                if (n + 3 < w.n && (w.n & 3) == 0) {
                    float4 o = make_float4(out[4 * q] + mid[4 * q], out[4 * q + 1] + mid[4 * q + 1], out[4 * q + 2] + mid[4 * q + 2],
                                           out[4 * q + 3] + mid[4 * q + 3]);
                    float4* p = reinterpret_cast<float4*>(yr + n);
                    if (!first) {
                        const float4 z = *p;
                        o = make_float4(add3(z.x, out[4 * q], mid[4 * q]), add3(z.y, out[4 * q + 1], mid[4 * q + 1]),
                                        add3(z.z, out[4 * q + 2], mid[4 * q + 2]), add3(z.w, out[4 * q + 3], mid[4 * q + 3]));
                    }
                    *p = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (n + e < w.n)
                            yr[n + e] = first ? out[4 * q + e] + mid[4 * q + e] : add3(yr[n + e], out[4 * q + e], mid[4 * q + e]);
                }
            }
        }
    };

    issue(0, 0);
    if (Y::kSlots == 3) issue(1, 1);
    uint32_t slot = 0;
    auto step = [&](uint32_t s) __attribute__((always_inline)) {
        // step s has landed, and every wavefront is past step s - 1, whose slot is filled next
        if (Y::kSlots == 3) wait_vm_n(nd);
        else wait_vm<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (Y::kSlots == 3) issue(s + 2, slot == 0 ? 2 : slot - 1);
        else issue(s + 1, slot ^ 1);
        const uint8_t* bs = lds + slot * Y::kBSlot + rh * 8192 + lane * 16;
        const uint8_t* ds = lds + slot * Y::kBSlot + Y::kSc + rh * 2048 + lane * 8;
        const uint8_t* ws = lds + Y::kOffW + slot * Y::kWSlot + cw * T::kSlot;
        Scales<DT> S;
        read_scales<DT, DV>(S, w, ws, nullptr, col0, lane, s, nch);
        uint2 ms = make_uint2(0, 0);
        if constexpr (T::kMin32) ms = *reinterpret_cast<const uint2*>(lds + slot * Y::kBSlot + Y::kMs + rh * 512 + lane * 8);
        // chunk j's products are issued, then chunk j + 1 is expanded beside them, then
        // chunk j is folded
        f16v t;
        h8 A[2][2];
        Bytes by;
        uint4 b[2];
        uint2 bd;
        auto read_b = [&](int j) {
            b[0] = *reinterpret_cast<const uint4*>(bs + j * 2048);
            b[1] = *reinterpret_cast<const uint4*>(bs + j * 2048 + 1024);
            bd = *reinterpret_cast<const uint2*>(ds + j * 512);
        };
        read_chunk<DT>(by, ws, lrow, 0, g);
        read_b(0);
        expand<DT>(by, 0, g, S, A[0]);
        read_chunk<DT>(by, ws, lrow, 1, g);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            Unit<DT> un;
            unit_mma<DT>(un, A[j & 1], S, j, b, bd, T::kMin32 ? chunk_sum(ms, j) : ms);
            __builtin_amdgcn_sched_barrier(0);
            if (j < 3) {
                read_b(j + 1);
                expand<DT>(by, j + 1, g, S, A[(j + 1) & 1]);
                asm volatile("" : "+v"(A[(j + 1) & 1][0]), "+v"(A[(j + 1) & 1][1]));
                if (j < 2) read_chunk<DT>(by, ws, lrow, j + 2, g);
            }
            __builtin_amdgcn_sched_barrier(0);
            unit_add<DT>(un, j == 0, t);
            asm volatile("" : "+v"(t));  // folded here, not at the step's end (four chunks' sums would not fit)
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int e = 0; e < 16; e++) mid[e] += t[e];
        slot = slot + 1 == Y::kSlots ? 0 : slot + 1;
    };
    // Steps summed in mid, and between two stores of the tile (even shares of at most 16).
    // So the relative L2 error against exact sums is no larger than the matvec kernels',
    // theirs / this: Q4_0 K = 1024 6.6e-8 / 6.3e-8, 2560 7.2e-8 / 6.9e-8, 4096 7.4e-8 /
    // 7.3e-8, 14336 8.4e-8 / 8.3e-8.  Q4_1's has one rounding a block more to make up
    // for, which takes shorter chains over a short K (7.65e-8 / 7.54e-8 at 4096 with,
    // 7.71e-8 without; 348 against 325 us at m = 512 4096 -> 14336).
    const uint32_t fold = DT == XNQ_Q4_1 && nstep < 24 ? 2 : 4;
    const uint32_t most = DT == XNQ_Q4_1 && nstep <= 40 ? 2 * fold : 16, stores = (nstep + most - 1) / most;
    const uint32_t share = (nstep + stores * fold - 1) / (stores * fold) * fold;
    for (uint32_t s16 = 0; s16 < nstep; s16 += share) {
        const uint32_t e16 = min(s16 + share, nstep);
        out = f16v{};
        for (uint32_t s4 = s16; s4 < e16; s4 += fold) {
            const uint32_t e4 = min(s4 + fold, e16);
            mid = f16v{};
            for (uint32_t s = s4; s < e4; s++) step(s);
            if (e4 == e16) break;
#pragma unroll
            for (int e = 0; e < 16; e++) out[e] += mid[e];
        }
        flush(s16 == 0);
    }
    wait_vm<0>();  // no DMA outlives the workgroup's LDS
}

template <int DT, int TM, bool DV, bool ROWS = false>
hipError_t launch_ksplit(const WView& w, const AView& a, size_t m, float* y, hipStream_t s) {
    using T = HT<DT>;
    constexpr int kWaveLds = 3 * T::kSlot + T::kDl, kRed = kWaves * TM * 4 * 64 * 16;
    constexpr int kLds = kWaves * kWaveLds > kRed ? kWaves * kWaveLds : kRed;
    const hipError_t e = set_max_lds(reinterpret_cast<const void*>(h16_ksplit_kernel<DT, TM, DV, ROWS>), kLds);
    if (e != hipSuccess) return e;
    const uint32_t n_tiles = (w.n + 31) / 32, rts = (uint32_t)((m + 31) / 32), m_tiles = (rts + TM - 1) / TM;
    const uint32_t grid = (m_tiles * n_tiles + 7) / 8 * 8;
    h16_ksplit_kernel<DT, TM, DV, ROWS><<<grid, kThreads, kLds, s>>>(w, a, (uint32_t)m, m_tiles, n_tiles, y);
    return hipGetLastError();
}

template <int DT>
hipError_t launch_ksplit16(const WView& w, const AView& a, size_t m, float* y, hipStream_t s) {
    constexpr int kWaveLds = 3 * HT<DT>::kSlot, kRed = kWaves * 2 * 64 * 16;
    constexpr int kLds = kWaves * kWaveLds > kRed ? kWaves * kWaveLds : kRed;
    const hipError_t e = set_max_lds(reinterpret_cast<const void*>(h16_ksplit16_kernel<DT>), kLds);
    if (e != hipSuccess) return e;
    const uint32_t n_tiles = (w.n + 31) / 32, m_tiles = (uint32_t)((m + 15) / 16);
    const uint32_t grid = (m_tiles * n_tiles + 7) / 8 * 8;
    h16_ksplit16_kernel<DT><<<grid, kThreads, kLds, s>>>(w, a, (uint32_t)m, m_tiles, n_tiles, y);
    return hipGetLastError();
}

// The kernel of m rows by n columns: 16-, 32- or 64-row tiles with K split over the
// wavefronts, or 256 x 64 tiles.
enum class Form { kSplit16, kSplit32, kSplit64, kTile };

// From the row images: 32-row tiles up to one workgroup per CU, then 64-row ones.
Form rows_form(size_t m, size_t n) {
    const size_t rts = (m + 31) / 32, n32 = (n + 31) / 32;
    return rts == 1 || rts * n32 <= 256 ? Form::kSplit32 : Form::kSplit64;
}

template <int DT, bool DV>
Form h16_form(size_t m, size_t n) {
    const size_t n32 = (n + 31) / 32;
    if (!HT<DT>::kK && DV) {
        // 16-row tiles up to one workgroup per CU (two rounds of them against one of
        // 32-row tiles: Q8_0 N = 4096 m = 64 19.3 / 14.7), and where 32 rows would be half
        // padding.  Not where planed scales do not come with the stage (K % 128 != 0):
        // loads of their own inside it lose (Q8_0 1056 -> 2048 m = 48 9.1 / 8.2)
        if (m <= 16 || (m + 15) / 16 * n32 <= 256) return Form::kSplit16;
    }
    // 32-row tiles up to one workgroup per CU, then 64-row tiles (Q8_0, K = 4096, us, graph
    // steps: N = 1024 m = 256 17 / 21, 512 31 / 25; N = 4096 m = 64 15 / 19, 128 25 / 21)
    if (rows_form(m, n) == Form::kSplit32) return Form::kSplit32;
    // A round of 256 x 64 tiles (one a CU) costs the same however few it holds; a round
    // of 64-row K-split workgroups is the products of 32 tiles.  So the tile pays from
    // so many K-split rounds, us, K = N = 4096, K-split / tile: Q2K m = 256 (2 rounds)
    // 40 / 52, 320 (3) 59 / 52; Q5K 384 (3) 46 / 54, 448 (4) 58 / 55; Q3K 384 42 / 52,
    // 512 (4) 54 / 52; Q8_0 512 (4) 66 / 67, 576 (5) 81 / 68; Q4_0 512 65 / 70, 576
    // 79 / 70; Q5_0 640 (5) 80 / 92, 768 (6) 97 / 93; scales not staged (Q8_0, K = 4160) 640
    // 88 / 103.  Q4_1's and Q5_1's lines were drawn when their 64-row K-split kernels spilled (512
    // 140 / 141, 640 133 / 135); these are the faster ones now up to 8 rounds (Q4_1 576 93 / 146,
    // 1024 157 / 174; Q5_1 704 103 / 139, 1024 149 / 152), except Q5_1 over a short K (K = 1024
    // 768 43 / 43, 1024 56 / 47), and the lines have not been drawn anew.
    constexpr size_t kRounds = DT == XNQ_Q2K ? 2 : DT == XNQ_Q5K ? 3 : DT == XNQ_Q5_0 || DT == XNQ_Q5_1 || !DV ? 5 : 4;
    const size_t tiles = ((m + 63) / 64) * ((n + 255) / 256), rounds = (tiles + 255) / 256;
    return tiles <= rounds * kRounds * 32 ? Form::kSplit64 : Form::kTile;
}

template <int DT, bool DV>
hipError_t launch_rows_dt(const WView& w, const AView& a, size_t m, float* y, hipStream_t s) {
    if (rows_form(m, w.n) == Form::kSplit32) return launch_ksplit<DT, 1, DV, true>(w, a, m, y, s);
    return launch_ksplit<DT, 2, DV, true>(w, a, m, y, s);
}

template <int DT, bool DV>
hipError_t launch_h16_dt(const WView& w, const AView& a, size_t m, float* y, hipStream_t s) {
    const Form f = h16_form<DT, DV>(m, w.n);
    if constexpr (!HT<DT>::kK && DV)
        if (f == Form::kSplit16) return launch_ksplit16<DT>(w, a, m, y, s);
    if (f == Form::kSplit32) return launch_ksplit<DT, 1, DV>(w, a, m, y, s);
    if (f == Form::kSplit64) return launch_ksplit<DT, 2, DV>(w, a, m, y, s);
    const uint32_t m_tiles = (uint32_t)((m + 63) / 64), n_tiles = (w.n + 255) / 256, grid = (m_tiles * n_tiles + 7) / 8 * 8;
    if constexpr (HT<DT>::kK) {
        constexpr int kLds = TLay<DT>::kLds;
        const hipError_t e = set_max_lds(reinterpret_cast<const void*>(h16_super_tile_kernel<DT>), kLds);
        if (e != hipSuccess) return e;
        h16_super_tile_kernel<DT><<<grid, kThreads, kLds, s>>>(w, a, (uint32_t)m, m_tiles, n_tiles, y);
    } else {
        constexpr int kLds = BLay<DT>::kLds;
        const hipError_t e = set_max_lds(reinterpret_cast<const void*>(h16_block_tile_kernel<DT, DV>), kLds);
        if (e != hipSuccess) return e;
        h16_block_tile_kernel<DT, DV><<<grid, 1024, kLds, s>>>(w, a, (uint32_t)m, m_tiles, n_tiles, y);
    }
    return hipGetLastError();
}

}  // namespace

bool h16_supported(uint32_t dtype) {
    return dtype == XNQ_Q8_0 || dtype == XNQ_Q4_0 || is_raw_layout(dtype);
}

// f(type, whether the scales come with the stage) of a weight of type dt and nb blocks a row
template <class F>
static auto by_type(uint32_t dt, size_t nb, F f) {
    using std::integral_constant;
    switch (dt) {
    case XNQ_Q8_0:
        return nb % 4 == 0 ? f(integral_constant<int, XNQ_Q8_0>{}, std::true_type{})
                           : f(integral_constant<int, XNQ_Q8_0>{}, std::false_type{});
    case XNQ_Q4_0:
        return nb % 4 == 0 ? f(integral_constant<int, XNQ_Q4_0>{}, std::true_type{})
                           : f(integral_constant<int, XNQ_Q4_0>{}, std::false_type{});
    case XNQ_Q4_1: return f(integral_constant<int, XNQ_Q4_1>{}, std::true_type{});
    case XNQ_Q5_0: return f(integral_constant<int, XNQ_Q5_0>{}, std::true_type{});
    case XNQ_Q5_1: return f(integral_constant<int, XNQ_Q5_1>{}, std::true_type{});
    case XNQ_Q2K: return f(integral_constant<int, XNQ_Q2K>{}, std::true_type{});
    case XNQ_Q3K: return f(integral_constant<int, XNQ_Q3K>{}, std::true_type{});
    default: return f(integral_constant<int, XNQ_Q5K>{}, std::true_type{});  // Q5K (h16_supported types only)
    }
}

const char* h16_kernel(uint32_t dtype, size_t m, size_t n, size_t k) {
    const Form f = by_type(dtype, k / 32, [&](auto dt, auto dv) { return h16_form<dt.value, dv.value>(m, n); });
    if (f == Form::kTile) return is_kquant(dtype) ? "h16_super_tile" : "h16_block_tile";
    return f == Form::kSplit16 ? "h16_ksplit16" : f == Form::kSplit32 ? "h16_ksplit32" : "h16_ksplit64";
}

hipError_t launch_h16(const WView& w, const AView& a, size_t m, float* y, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    if (!a.h16 || (size_t)a.H.rts * 32 < m || a.k != w.k) return hipErrorInvalidValue;
    if (!h16_supported(w.dtype)) return hipErrorNotSupported;
    return by_type(w.dtype, w.nb, [&](auto dt, auto dv) { return launch_h16_dt<dt.value, dv.value>(w, a, m, y, s); });
}

hipError_t launch_h16_rows(const WView& w, const AView& a, size_t m, float* y, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    if (a.m < m || a.k != w.k) return hipErrorInvalidValue;
    if (!h16_supported(w.dtype)) return hipErrorNotSupported;
    return by_type(w.dtype, w.nb, [&](auto dt, auto dv) { return launch_rows_dt<dt.value, dv.value>(w, a, m, y, s); });
}

}  // namespace xnq
