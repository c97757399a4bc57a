// Dequant-fused product for a few activation rows (2..8) with the activations in REGISTERS:
// y[m, n] = sum_k x[m, k] * W[n, k] with every weight fetched once for all rows and no activation read from LDS.
//
// What bounds it: the weight bytes (0.5625 .. 1.0625 per weight); the arithmetic, one unpack per weight and four multiply-adds per
// MFMA, is about half of the VALU's time at that rate.  The other kernels for a few rows stage the activations in LDS, where
// a wave reads them again for every weight row (rows_stream_kernel: an operand per MFMA; the flat walk: four bytes per weight
// and f32 row) and where long rows of several activations do not fit.
//
// Mapping.  A workgroup works on groups of sixteen weight rows.  Its waves split k: wave w owns up to S super-blocks (256
// weights) of every row and keeps the activations that meet them as MFMA operands for the whole launch, 32 registers per
// super-block and sixteen columns.  bf16 rows are a column each, two of the four that a lane group's results are.  An f32 row is three columns: its value cut into three bf16
// parts of eight bits (all 24 bits of it, so the products are exact and only the f32 sums round); five rows make fifteen
// columns, six to eight rows two operands of twelve.  Per task -- one super-block of sixteen rows -- a wave copies the
// blocks from memory straight into a slot of LDS of its own (global_load_lds, consecutive lanes consecutive 16-byte pieces
// of a row), a ring of slots ahead of the arithmetic and with no barrier; lane (j, g) (j = lane % 16, g = lane / 16) then
// reads its eighth or sixteenth of row j's blocks, and the slot is refilled before the arithmetic starts.  The k parts meet in
// LDS once per group of rows, behind the only barrier of the loop, double-buffered.
//
// Weights enter the MFMA as small integers, exact in bf16.  The codes 0 .. 15 of an fp8 (e4m3) byte stand for that many 2^-9, its
// first binade and the subnormals below being one even ladder: a byte that holds a nibble IS the number, and
// v_cvt_scalef32_pk_bf16_fp8 makes two bf16 weights of two of them (1.9 ns per wave instruction, as much as one byte permute or and-or; a
// conversion per weight and a permute per pair take 2.7 times as long, a nibble under the bits of 16.0 as long but its sums lose
// two bits to the 16).  The fifth bit of Q5_K and the upper two of Q6_K are numbers of their own in a second MFMA chained to the
// first, with the format's -32 in it (-2 .. 1 times 16).  Q8_0: signed bytes, converted.  Q4_0's -8 likewise.  The mins of Q4_K and Q5_K leave
// through the sub-blocks' activation sums in a small f32 MFMA.
#pragma once

#include <type_traits>

#include "gemvk_plan.h"
#include "hq_internal.h"

namespace hq {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr uint32_t kKMaxSegs = 4;
struct KRowsArgs {
    const void* x;           // row r, element e at r * xstride + e; heads outermost (hd != 0): at (e / hd) * xplane + r * xstride + e % hd
    uint32_t xstride, hd, xplane;
    uint32_t m, k, rowb;     // rowb: bytes of a weight row
    uint32_t sb0, nsb;       // the launch covers super-blocks sb0 .. sb0 + nsb - 1 of every row
    uint32_t kp, rg, ring;   // waves that share a group's k, groups side by side in a workgroup, slots of a wave's ring
    uint32_t base, extra;    // super-blocks per wave: nsb / kp, and the first nsb % kp waves one more
    uint32_t units, full, rem;  // groups of sixteen rows, all segments (swiglu: of one matrix); units over gridDim * rg, and the rest
    uint32_t whole;          // sums are taken again where they are infinite or NaN
    const float* gate;       // may be null, laid out as y[0]: silu(gate) * product is stored
    uint32_t add, swiglu;    // add: products are added to y; swiglu: seg 0 = gate, seg 1 = up, y[0] = silu(gate) * up
    uint32_t nseg;
    const uint8_t* w[kKMaxSegs];
    float* y[kKMaxSegs];
    uint32_t n[kKMaxSegs], end[kKMaxSegs];  // rows of a segment, the first group past it
};

namespace {

__device__ __forceinline__ f32x4_t mfma32(const uint4& a, const uint4& b, const f32x4_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma16(uint32_t a0, uint32_t a1, const uint2& b, const f32x4_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4_t, make_uint2(a0, a1)), __builtin_bit_cast(bf16x4_t, b), c, 0, 0, 0);
}
// Four bytes of fp8 codes 0 .. 15 (or 0x81 .. for negative numbers) as four bf16 numbers times scale / 512.
__device__ __forceinline__ uint2 from_codes(uint32_t w, float scale) {
    return make_uint2(__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, false)),
                      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, true)));
}
__device__ __forceinline__ uint4 from_codes(uint32_t w0, uint32_t w1, float scale) {
    const uint2 a = from_codes(w0, scale), b = from_codes(w1, scale);
    return make_uint4(a.x, a.y, b.x, b.y);
}
constexpr float kOne = 512.f, kSixteen = 8192.f;
constexpr uint32_t N4 = 0x0f0f0f0fu, N2 = 0x03030303u, N1 = 0x01010101u;
constexpr f32x4_t kZero = {0.f, 0.f, 0.f, 0.f};

// The activations of one super-block as operands: a[i] = the lane's eight activations of sub-block i (Q6_K: two groups of
// four, of scale groups 2 i and 2 i + 1); s[t] = the activation sum of sub-block 4 t + g, the lane's entry of the small f32 MFMA.
template <int NSUM>
struct XFrag {
    uint4 a[8];
    float s[NSUM ? NSUM : 1];
};

template <int TYPE>
struct KWeights;

// Q4_K / Q5_K: lane (j, g) takes bytes 8 g .. 8 g + 7 of each chunk of 32 nibble bytes: sub-blocks 2 c (low nibbles) and 2 c + 1.
template <bool Q5>
struct KWeightsQ45 {
    static constexpr uint32_t BYTES = Q5 ? Q5K_BYTES : Q4K_BYTES, QS = Q5 ? 48u : 16u;
    static constexpr uint32_t NEED = BYTES / 16u, PITCH = NEED;  // 16-byte pieces of a block, and of a row of a slot (odd: sixteen groups of four banks)
    static constexpr int NSUM = 2;
    static constexpr bool G16 = false;
    uint4 hdr;
    uint2 q[4], qh;
    __device__ __forceinline__ void read(const uint8_t* p, uint32_t g, uint32_t) {
        hdr = *reinterpret_cast<const uint4*>(p);
        if constexpr (Q5) qh = *reinterpret_cast<const uint2*>(p + 16u + 8u * g);
#pragma unroll
        for (int c = 0; c < 4; ++c) q[c] = *reinterpret_cast<const uint2*>(p + QS + 8u * g + 32 * c);
    }
    template <int NF, int NV>
    __device__ __forceinline__ void mul(const XFrag<NSUM> (&x)[NF], uint32_t g, f32x4_t (&acc)[NF]) const {
        // (the codes stand for 2^-10 of their number and d for 2^10 of its own: a sum of a sub-block times its six bits of scale is no larger than
        // its activations allow, and overflows no earlier than the product does)
        const float d = 1024.f * f16_bits_to_f32(hdr.x & 0xffffu), dmin = f16_bits_to_f32(hdr.x >> 16);
        const uint32_t zs = hdr.z >> (8u * g), ws = hdr.w >> (8u * g);
        // mins of sub-blocks g and 4 + g
        const float o0 = dmin * (float)(zs & 63u), o1 = dmin * (float)(((ws >> 4) & 15u) | ((zs >> 2) & 0x30u));
        const uint32_t sl = hdr.y & 0x3f3f3f3fu, sh = (hdr.w & N4) | ((hdr.y >> 2) & 0x30303030u);
        f32x4_t t[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[f].s[0], -o0, acc[f], 0, 0, 0);
            acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[f].s[1], -o1, acc[f], 0, 0, 0);
            t[f] = kZero;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t s = c < 2 ? sl : sh;
            const float s0 = c & 1 ? ubyte2(s) : ubyte0(s), s1 = c & 1 ? ubyte3(s) : ubyte1(s);
            const uint4 lo = from_codes(q[c].x & N4, q[c].y & N4, kOne / 1024.f), hi = from_codes((q[c].x >> 4) & N4, (q[c].y >> 4) & N4, kOne / 1024.f);
            uint4 lo5, hi5;
            if constexpr (Q5) {
                lo5 = from_codes((qh.x >> (2 * c)) & N1, (qh.y >> (2 * c)) & N1, kSixteen / 1024.f);
                hi5 = from_codes((qh.x >> (2 * c + 1)) & N1, (qh.y >> (2 * c + 1)) & N1, kSixteen / 1024.f);
            }
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const f32x4_t a = mfma32(x[f].a[2 * c], lo, Q5 ? mfma32(x[f].a[2 * c], lo5, kZero) : kZero);
                const f32x4_t b = mfma32(x[f].a[2 * c + 1], hi, Q5 ? mfma32(x[f].a[2 * c + 1], hi5, kZero) : kZero);
#pragma unroll
                for (int v = 0; v < NV; ++v) t[f][v] = fmaf(s1, b[v], fmaf(s0, a[v], t[f][v]));
            }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[f][v] = fmaf(d, t[f][v], acc[f][v]);
    }
};
template <>
struct KWeights<HQ_Q4_K> : KWeightsQ45<false> {};
template <>
struct KWeights<HQ_Q5_K> : KWeightsQ45<true> {};

// Q6_K: scales cover sixteen weights, MFMAs of k = 16; lane (j, g) takes weights 4 g .. 4 g + 3 of a group.  A block is
// 210 bytes: rows of a slot start at the 16-byte boundary below their block, and the lane shifts its words into place.
template <>
struct KWeights<HQ_Q6_K> {
    static constexpr uint32_t BYTES = Q6K_BYTES, NEED = 14u, PITCH = 15u;
    static constexpr int NSUM = 0;
    static constexpr bool G16 = true;
    uint32_t ql[8], qh[4], sc[4];
    float d;
    __device__ __forceinline__ void read(const uint8_t* p, uint32_t g, uint32_t mis) {
        const uint32_t odd = mis & 2u;
        p += mis - odd;
        const uint32_t* b = reinterpret_cast<const uint32_t*>(p) + g;
        uint32_t lo[12], hi[12], t[5];
#pragma unroll
        for (int i = 0; i < 12; ++i) {  // ql: h u s -> bytes 64 h + 32 u + 16 s; qh: h s -> 128 + 32 h + 16 s
            const int off = i < 8 ? 16 * (i >> 2) + 8 * ((i >> 1) & 1) + 4 * (i & 1) : 32 + 8 * ((i - 8) >> 1) + 4 * (i & 1);
            lo[i] = b[off], hi[i] = b[off + 1];
        }
        const uint32_t* e = reinterpret_cast<const uint32_t*>(p) + 48;
#pragma unroll
        for (int i = 0; i < 5; ++i) t[i] = e[i];
#pragma unroll
        for (int i = 0; i < 12; ++i) (i < 8 ? ql[i] : qh[i - 8]) = __builtin_amdgcn_alignbyte(hi[i], lo[i], odd);
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[i] = __builtin_amdgcn_alignbyte(t[i + 1], t[i], odd);
        d = f16_bits_to_f32((t[4] >> (8u * odd)) & 0xffffu);
        // (shifted here: kept as read, the words would take twice the registers)
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(ql[i]));
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(qh[i]), "+v"(sc[i]));
    }
    template <int NF, int NV>
    __device__ __forceinline__ void mul(const XFrag<NSUM> (&x)[NF], uint32_t, f32x4_t (&acc)[NF]) const {
        constexpr uint32_t SIGNED2 = 0x01008182u;  // fp8 codes of -2, -1, 0, 1 by their two bits
        f32x4_t t[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) t[f] = kZero;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t hq = qh[2 * h + s];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t w = ql[4 * h + 2 * (r & 1) + s];
                    const uint2 lo = from_codes((r >= 2 ? w >> 4 : w) & N4, kOne);
                    const uint2 hi = from_codes(__builtin_amdgcn_perm(SIGNED2, SIGNED2, (hq >> (2 * r)) & N2), kSixteen);
                    const int G = 8 * h + 2 * r + s;
                    const float scale = sbyte(sc[G >> 2], G & 3);
#pragma unroll
                    for (int f = 0; f < NF; ++f) {
                        const uint4& av = x[f].a[G >> 1];
                        const uint32_t a0 = G & 1 ? av.z : av.x, a1 = G & 1 ? av.w : av.y;
                        const f32x4_t c = mfma16(a0, a1, lo, mfma16(a0, a1, hi, kZero));
#pragma unroll
                        for (int v = 0; v < 4; ++v) t[f][v] = fmaf(scale, c[v], t[f][v]);
                    }
                }
                // (four groups at a time: left to itself the compiler keeps the results of all sixteen MFMAs ahead of the sums)
#pragma unroll
                for (int f = 0; f < NF; ++f) asm volatile("" : "+v"(t[f]));
            }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[f][v] = fmaf(d, t[f][v], acc[f][v]);
    }
};

// Eight 32-weight blocks of Q8_0 (272 bytes) or Q4_0 (144) stand for a super-block.  A block starts at an even address: for even
// blocks three aligned words are shifted into place.
template <uint32_t BB>
struct KBlocks32 {
    static constexpr uint32_t BYTES = 8u * BB, NEED = BYTES / 16u, PITCH = NEED;
    uint2 q[8];
    uint32_t d[8];
    // off: the lane's eight bytes within a block's quants (a multiple of four)
    __device__ __forceinline__ void read_at(const uint8_t* p, uint32_t off) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (c & 1) {
                const uint32_t* w = reinterpret_cast<const uint32_t*>(p + BB * c + 2u + off);
                q[c] = make_uint2(w[0], w[1]);
                d[c] = *reinterpret_cast<const uint32_t*>(p + BB * c - 2u) >> 16;
            } else {
                const uint32_t* w = reinterpret_cast<const uint32_t*>(p + BB * c + off);
                const uint32_t a0 = w[0], a1 = w[1], a2 = w[2];
                q[c] = make_uint2(__builtin_amdgcn_alignbyte(a1, a0, 2), __builtin_amdgcn_alignbyte(a2, a1, 2));
                d[c] = *reinterpret_cast<const uint32_t*>(p + BB * c) & 0xffffu;
            }
        }
    }
};
template <>
struct KWeights<HQ_Q8_0> : KBlocks32<Q8_0_BYTES> {
    static constexpr int NSUM = 0;
    static constexpr bool G16 = false;
    __device__ __forceinline__ void read(const uint8_t* p, uint32_t g, uint32_t) { read_at(p, 8u * g); }
    static __device__ __forceinline__ uint32_t pair(uint32_t w, int lo) {  // small integers: their upper halves are the bf16 values
        return __builtin_amdgcn_perm(__float_as_uint(sbyte(w, lo + 1)), __float_as_uint(sbyte(w, lo)), 0x07060302u);
    }
    template <int NF, int NV>
    __device__ __forceinline__ void mul(const XFrag<NSUM> (&x)[NF], uint32_t, f32x4_t (&acc)[NF]) const {
        f32x4_t t[NF][2];  // (the two halves' sums apart: fewer roundings in a row)
#pragma unroll
        for (int f = 0; f < NF; ++f) t[f][0] = t[f][1] = kZero;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float dc = f16_bits_to_f32(d[c]);
            const uint4 b = make_uint4(pair(q[c].x, 0), pair(q[c].x, 2), pair(q[c].y, 0), pair(q[c].y, 2));
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const f32x4_t r = mfma32(x[f].a[c], b, kZero);
#pragma unroll
                for (int v = 0; v < NV; ++v) t[f][c / 4][v] = fmaf(dc, r[v], t[f][c / 4][v]);
            }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[f][v] += t[f][0][v] + t[f][1][v];
    }
};
// Q4_0: lane group g takes the low (g < 2) or high nibbles of bytes 8 (g & 1) .. + 7.  q - 8 is the lower three bits, and -8 where the
// fourth is clear, in a second MFMA (as sums of q and of the activations the products would lose two bits to the 8).
template <>
struct KWeights<HQ_Q4_0> : KBlocks32<Q4_0_BYTES> {
    static constexpr int NSUM = 0;
    static constexpr bool G16 = false;
    __device__ __forceinline__ void read(const uint8_t* p, uint32_t g, uint32_t) { read_at(p, 8u * (g & 1u)); }
    static __device__ __forceinline__ uint32_t minus8(uint32_t w) {  // the code of -8 in the bytes whose fourth bit is clear
        const uint32_t t = ~w & 0x08080808u;
        return t << 4 | t;
    }
    template <int NF, int NV>
    __device__ __forceinline__ void mul(const XFrag<NSUM> (&x)[NF], uint32_t g, f32x4_t (&acc)[NF]) const {
        const uint32_t sh = 4u * (g >> 1);
        f32x4_t t[NF][2];
#pragma unroll
        for (int f = 0; f < NF; ++f) t[f][0] = t[f][1] = kZero;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float dc = f16_bits_to_f32(d[c]);
            const uint32_t w0 = q[c].x >> sh, w1 = q[c].y >> sh;
            const uint4 b = from_codes(w0 & 0x07070707u, w1 & 0x07070707u, kOne), b8 = from_codes(minus8(w0), minus8(w1), kOne);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const f32x4_t r = mfma32(x[f].a[c], b, mfma32(x[f].a[c], b8, kZero));
#pragma unroll
                for (int v = 0; v < NV; ++v) t[f][c / 4][v] = fmaf(dc, r[v], t[f][c / 4][v]);
            }
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[f][v] += t[f][0][v] + t[f][1][v];
    }
};

// The three bf16 parts of x, each the upper half of the f32 it stands for: eight bits each, cut and not rounded, so that the
// three add up to x and none overflows.  An infinity or NaN has to be its first part alone (CHECK); `nan` becomes NaN where one was met.
template <bool CHECK>
__device__ __forceinline__ void bf16_parts(uint32_t u, uint32_t (&p)[3], float& nan) {
    const bool fin = !CHECK || (u & 0x7f800000u) != 0x7f800000u;
    p[0] = (u & 0xffff0000u) | (CHECK && !fin && (u & 0x007fffffu) ? 0x00400000u : 0u);
    const float r = fin ? __uint_as_float(u) - __uint_as_float(p[0]) : 0.f;
    if (!CHECK) nan = fmaf(r, 0.f, nan);
    p[1] = __float_as_uint(r) & 0xffff0000u;
    p[2] = __float_as_uint(r - __uint_as_float(p[1]));
}

// Columns.  Value v of lane group g of an MFMA's result is column 4 g + v, and only the first NV values of a group are used, so
// that the sums per sub-block cost NV multiply-adds: bf16 rows (NV 2) r = 2 g + v; f32 rows: operand f holds the rows from f * krows_per
// on, part g of row v in column 4 g + v (g < 3), and where it holds NV + 1 rows the last one's part v in column 12 + v.
__device__ __forceinline__ uint32_t krows_per(uint32_t m, int nf) { return nf == 2 ? (m + 1u) / 2u : m; }

// The activation rows of a super-block as they lie in memory: a lane has four of each row.
template <bool F32, int NV, int NF>
struct XRows {
    static constexpr int N = F32 ? NV + 1 : 8;  // rows of an operand
    uint4 r[NF][F32 ? N : N / 2];               // (bf16: two rows to a uint4)
    __device__ __forceinline__ void load(const KRowsArgs& a, uint32_t k0, uint32_t lane) {
        const uint32_t per = krows_per(a.m, NF), kk = k0 + 4u * lane;
        const size_t at = a.hd ? (size_t)(kk / a.hd) * a.xplane + kk % a.hd : kk;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int i = 0; i < N; ++i)
                if ((uint32_t)i < per && f * per + i < a.m) {
                    const size_t e = (size_t)(f * per + i) * a.xstride + at;
                    if constexpr (F32) {
                        r[f][i] = *reinterpret_cast<const uint4*>(static_cast<const float*>(a.x) + e);
                    } else {
                        const uint2 t = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.x) + e);
                        if (i & 1) r[f][i / 2].z = t.x, r[f][i / 2].w = t.y;
                        else r[f][i / 2].x = t.x, r[f][i / 2].y = t.y;
                    }
                }
    }
    __device__ __forceinline__ void arrived() {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int i = 0; i < (F32 ? N : N / 2); ++i) asm volatile("" : "+v"(r[f][i].x), "+v"(r[f][i].y), "+v"(r[f][i].z), "+v"(r[f][i].w));
    }
};

// A super-block's activations as operands: rows are cut into their parts once and handed to the lanes that want them through `tmp`, 2112
// bytes of LDS of the wave's own, up to four columns at a time.
constexpr uint32_t kXPitch = 528;  // bytes from a column to the next
template <bool F32, int NV, int NF, int NSUM, bool G16>
__device__ __forceinline__ void make_frags(XFrag<NSUM> (&x)[NF], const XRows<F32, NV, NF>& raw, const KRowsArgs& a, uint32_t lane, uint8_t* tmp) {
    const uint32_t c = lane & 15u, g = lane >> 4, cg = c >> 2, cv = c & 3u;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 8; ++i) x[f].a[i] = make_uint4(0, 0, 0, 0);
    // the lane's operands out of 256 bf16 activations of one column
    auto take = [&](XFrag<NSUM>& fr, const uint8_t* col) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (G16) {
                const uint2 lo = *reinterpret_cast<const uint2*>(col + 64 * i + 8u * g), hi = *reinterpret_cast<const uint2*>(col + 64 * i + 32 + 8u * g);
                fr.a[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            } else {
                fr.a[i] = *reinterpret_cast<const uint4*>(col + 64 * i + 16u * g);
            }
        }
    };
    if constexpr (!F32) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {  // rows 4 p .. 4 p + 3
            if (4u * p >= a.m) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4& t = raw.r[0][2 * p + i / 2];
                *reinterpret_cast<uint2*>(tmp + i * kXPitch + 8u * lane) = i & 1 ? make_uint2(t.z, t.w) : make_uint2(t.x, t.y);
            }
            asm volatile("" ::: "memory");  // (one wave's LDS instructions are served in order)
            const uint32_t row = 2u * cg + cv;
            if (cv < 2u && row >> 2 == (uint32_t)p && row < a.m) take(x[0], tmp + (row & 3u) * kXPitch);
            asm volatile("" ::: "memory");
        }
    } else {
        const uint32_t per = krows_per(a.m, NF);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            uint2 w[NV + 1][3];
            float nan = 0.f;
            auto cut = [&](auto check) {
                constexpr bool CHECK = decltype(check)::value;
#pragma unroll
                for (int i = 0; i < NV + 1; ++i)
                    if ((uint32_t)i < per && f * per + i < a.m) {
                        uint32_t e[4][3];
                        bf16_parts<CHECK>(raw.r[f][i].x, e[0], nan);
                        bf16_parts<CHECK>(raw.r[f][i].y, e[1], nan);
                        bf16_parts<CHECK>(raw.r[f][i].z, e[2], nan);
                        bf16_parts<CHECK>(raw.r[f][i].w, e[3], nan);
#pragma unroll
                        for (int p = 0; p < 3; ++p)
                            w[i][p] = make_uint2(__builtin_amdgcn_perm(e[1][p], e[0][p], 0x07060302u), __builtin_amdgcn_perm(e[3][p], e[2][p], 0x07060302u));
                    }
            };
            cut(std::false_type{});
            if (__any(nan != nan)) cut(std::true_type{});
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t cols = p == 3 ? (per == NV + 1u && f * per + NV < a.m ? 3u : 0u) : per < (uint32_t)NV ? per : (uint32_t)NV;
#pragma unroll
                for (int i = 0; i < (p == 3 ? 3 : NV); ++i)
                    if (p == 3 ? cols != 0u : (uint32_t)i < per && f * per + i < a.m)
                        *reinterpret_cast<uint2*>(tmp + i * kXPitch + 8u * lane) = p == 3 ? w[NV][i] : w[i][p % 3];
                asm volatile("" ::: "memory");
                if (cg == (uint32_t)p && cv < cols && (p == 3 || f * per + cv < a.m)) take(x[f], tmp + cv * kXPitch);
                asm volatile("" ::: "memory");
            }
        }
    }
    if constexpr (NSUM) {
        constexpr uint32_t ONES = 0x3f803f80u;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int t = 0; t < NSUM; ++t) {
                float s[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint4& v = x[f].a[4 * t + i];
                    s[i] = dot2_bf16(v.w, ONES, dot2_bf16(v.z, ONES, dot2_bf16(v.y, ONES, dot2_bf16(v.x, ONES, 0.f))));
                    s[i] = xor32_add(xor16_add(s[i]));
                    asm volatile("" : "+v"(s[i]));
                }
                const float lo = g & 1u ? s[1] : s[0], hi = g & 1u ? s[3] : s[2];
                x[f].s[t] = g & 2u ? hi : lo;
            }
    }
}

template <int NI>
__device__ __forceinline__ void wait_behind(uint32_t tasks) {  // all but the newest `tasks` tasks' fetches have landed
    if (tasks == 0u) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (tasks == 1u) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
    else if (tasks == 2u) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * NI) : "memory");
}
constexpr uint32_t kKMaxRing = 4;

// Weight e (of 256) of a super-block of Q4_0 or Q6_K.
template <int TYPE>
__device__ __forceinline__ float weight_at(const uint8_t* p, uint32_t e) {
    static_assert(TYPE == HQ_Q4_0 || TYPE == HQ_Q6_K, "the types of sum_again");
    if constexpr (TYPE == HQ_Q4_0) {
        p += Q4_0_BYTES * (e >> 5);
        const uint32_t q = p[2u + (e & 15u)];
        return f16_bits_to_f32(ld2(p)) * ((float)(e & 16u ? q >> 4 : q & 15u) - 8.f);
    } else {
        const uint32_t h = e >> 7, r = (e >> 5) & 3u, l = e & 31u, ql = p[64u * h + 32u * (r & 1u) + l], qh = p[128u + 32u * h + l];
        const float q = (float)((r >= 2u ? ql >> 4 : ql & 15u) | ((qh >> (2u * r)) & 3u) << 4) - 32.f;
        return f16_bits_to_f32(ld2(p + 208)) * (float)(int8_t)p[192u + (e >> 4)] * q;
    }
}

// A sum that came out infinite or NaN, once more with whole weights: row `row` of x and row lane % 16 of the group u, a lane group a quarter of
// k.  The MFMAs take a Q4_0 or Q6_K weight in two parts of opposite signs, for which an infinite activation is NaN even where the weight is not
// zero.  Where the row holds a NaN there is nothing to do, where it holds infinities their products are the sum, else all products (a
// part that was beyond f32).  The arguments are read here and not kept in registers.
typedef const __attribute__((address_space(4))) KRowsArgs* KRowsArgsPtr;
template <int TYPE, bool F32>
__device__ __forceinline__ float sum_again(uint32_t row, uint32_t u, uint32_t lane, uint32_t matrix) {
    uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(at), "+v"(lane));
    const KRowsArgsPtr a = (KRowsArgsPtr)at;
    const uint32_t k0 = a->sb0 * 256u, nsb = a->nsb, hd = a->hd;
    // a super-block's activations, four to a lane, as f32
    auto x4 = [&](uint32_t sb) {
        const uint32_t kk = k0 + sb * 256u + 4u * lane;
        const size_t i = (size_t)row * a->xstride + (hd ? (size_t)(kk / hd) * a->xplane + kk % hd : kk);
        if constexpr (F32) return *reinterpret_cast<const uint4*>(static_cast<const float*>(a->x) + i);
        const uint2 t = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a->x) + i);
        return make_uint4(t.x << 16, t.x & 0xffff0000u, t.y << 16, t.y & 0xffff0000u);
    };
    uint32_t most = 0;  // the largest magnitude, as bits: infinity 0x7f800000, NaNs above
#pragma unroll 4
    for (uint32_t sb = 0; sb < nsb; ++sb) {
        const uint4 v = x4(sb);
        const uint32_t ab = max(v.x & 0x7fffffffu, v.y & 0x7fffffffu), cd = max(v.z & 0x7fffffffu, v.w & 0x7fffffffu);
        most = max(most, max(ab, cd));
    }
    if (__any(most > 0x7f800000u)) return __builtin_nanf("");
    const bool odd = __any(most == 0x7f800000u);

    uint32_t seg = matrix, from = 0;
    if (!a->swiglu)
        while (seg + 1u < a->nseg && u >= a->end[seg]) from = a->end[seg++];
    const uint8_t* w = a->w[seg] + (size_t)((u - from) * 16u + (lane & 15u)) * a->rowb + (size_t)a->sb0 * KWeights<TYPE>::BYTES;
    float sum = 0.f;
#pragma unroll 1
    for (uint32_t sb = 0; sb < nsb; ++sb, w += KWeights<TYPE>::BYTES) {
        const uint4 v = x4(sb);
        auto inf = [](uint32_t b) { return (b & 0x7fffffffu) == 0x7f800000u; };
        uint64_t lanes = odd ? __ballot(inf(v.x) || inf(v.y) || inf(v.z) || inf(v.w)) : ~0ull;
        while (lanes) {  // lane l's four activations, one to each lane group
            const int l = __builtin_ctzll(lanes);
            lanes &= lanes - 1u;
            const uint32_t x0 = __builtin_amdgcn_readlane(v.x, l), x1 = __builtin_amdgcn_readlane(v.y, l), x2 = __builtin_amdgcn_readlane(v.z, l), x3 = __builtin_amdgcn_readlane(v.w, l);
            const uint32_t g = lane >> 4, x = g & 2u ? (g & 1u ? x3 : x2) : g & 1u ? x1 : x0;
            if (!odd || inf(x)) sum = fmaf(__uint_as_float(x), weight_at<TYPE>(w, 4u * l + g), sum);
        }
    }
    return xor32_add(xor16_add(sum));
}

// WHOLE: sums that are infinite or NaN are taken again (sum_again): where the kernel stands for a tile, whose weights are one number each, at nine to
// sixteen rows.  (The registers around that branch cost 1 to 2 %; the other kernels for two to eight rows take weights in parts as well.)
template <int TYPE, bool F32, int NV, int NF, int S, int W, bool WHOLE>
__global__ __launch_bounds__(64 * W) void krows_kernel(KRowsArgs a) {
    using T = KWeights<TYPE>;
    constexpr uint32_t PIECES = 16u * T::PITCH, SLOT = PIECES * 16u;
    constexpr int NI = (int)((PIECES + 63u) / 64u);
    static_assert((kKMaxRing - 1) * NI < 64, "the counter of outstanding loads");
    extern __shared__ uint4 smem4[];
    uint8_t* smem = reinterpret_cast<uint8_t*>(smem4);
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t j = lane & 15u, g = lane >> 4;
    const uint32_t waves = a.kp * a.rg, rgi = (wave >= a.kp) + (wave >= 2u * a.kp) + (wave >= 3u * a.kp), kw = wave - rgi * a.kp;  // (rg <= 4)
    const uint32_t cnt = a.base + (kw < a.extra ? 1u : 0u), first_sb = a.sb0 + kw * a.base + (kw < a.extra ? kw : a.extra);
    // groups: unit u of this wave in round r is (r * gridDim + block) * rg + rgi; with swiglu a round of gate, then one of up
    const uint32_t ustride = gridDim.x * a.rg, u0 = blockIdx.x * a.rg + rgi, shift = a.swiglu ? 1u : 0u;
    const uint32_t rounds_all = (a.full + (blockIdx.x * a.rg < a.rem ? 1u : 0u)) << shift, rounds = (a.full + (u0 < a.rem ? 1u : 0u)) << shift;

    // ---- the ring: fetches run ahead of the arithmetic by up to a.ring tasks ----
    uint8_t* slots = smem + (size_t)wave * a.ring * SLOT;
    const uint32_t slots_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)slots);
    uint32_t f_row[NI], f_off[NI];  // this lane's piece of fetch i: byte of its row in the group, byte in the row's pieces
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const uint32_t p = 64u * i + lane < PIECES ? 64u * i + lane : PIECES - 1u, r = p / T::PITCH, c = p - r * T::PITCH;
        f_row[i] = r * a.rowb;
        f_off[i] = 16u * (c < T::NEED ? c : T::NEED - 1u);
    }
    uint32_t f_left = rounds * cnt, f_s = 0, f_round = 0, f_slot = 0, f_u = u0, f_seg = 0;
    const size_t step = (size_t)ustride * 16u * a.rowb;
    const uint8_t* f_base = a.w[0] + (size_t)u0 * 16u * a.rowb;  // the group being fetched
    auto in_segment = [&]() {
        uint32_t from = f_seg ? a.end[f_seg - 1u] : 0u;
        if (f_u < a.end[f_seg]) return;
        while (f_seg + 1u < a.nseg && f_u >= a.end[f_seg]) from = a.end[f_seg++];
        f_base = a.w[f_seg] + (size_t)(f_u - from) * 16u * a.rowb;
    };
    auto fetch = [&]() {
        if (f_left == 0u) return;
        const uint32_t off = (first_sb + f_s) * T::BYTES, dst = slots_lds + f_slot * SLOT;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const uint32_t v = (T::BYTES % 16u ? (f_row[i] + off) & ~15u : f_row[i] + off) + f_off[i];
            // (inline assembly: the compiler would wait for every fetch into LDS ahead of any read from it; one wait state between a scalar write
            // of M0 and the load that reads it, which it does not put there)
            if (64u * (i + 1) <= PIECES || 64u * i + lane < PIECES)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(v), "s"(f_base), "s"(dst + 1024u * i) : "memory", "m0");
        }
        --f_left;
        if (++f_slot == a.ring) f_slot = 0;
        if (++f_s == cnt) {
            f_s = 0;
            ++f_round;
            if (a.swiglu) {
                f_base += f_round & 1u ? a.w[1] - a.w[0] : a.w[0] - a.w[1] + (ptrdiff_t)step;
            } else {
                f_u += ustride;
                f_base += step;
                if (f_left) in_segment();
            }
        }
    };
    if (!a.swiglu && f_left) in_segment();
    // The activations are waited for ahead of the first weights: loads return in order, and the arithmetic would begin behind the whole
    // ring otherwise.  They pass through the last slot, which is filled behind them.
    XFrag<T::NSUM> x[S][NF];
    {
        XRows<F32, NV, NF> raw[S];
#pragma unroll
        for (int s = 0; s < S; ++s)
            if ((uint32_t)s < cnt) raw[s].load(a, (first_sb + s) * 256u, lane);
#pragma unroll
        for (int s = 0; s < S; ++s) raw[s].arrived();
        for (uint32_t i = 1; i < a.ring; ++i) fetch();
#pragma unroll
        for (int s = 0; s < S; ++s)
            if ((uint32_t)s < cnt) make_frags<F32, NV, NF, T::NSUM, T::G16>(x[s], raw[s], a, lane, slots + (a.ring - 1u) * SLOT);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    fetch();
    T w;

    // ---- where the k parts meet: [buffer][group][k part][row][16] floats behind the rings ----
    float* red = reinterpret_cast<float*>(smem + (size_t)waves * a.ring * SLOT);
    const uint32_t part = a.m * 16u, buf = waves * part;
    // a wave adds up the parts of one activation row of one group: lane (j, g) those of k parts g, g + 4 ...  (from the last wave down:
    // those have a super-block less where nsb is no multiple of kp)
    const uint32_t rows_red = a.rg * a.m, wred = waves - 1u - wave;
    float held[2] = {0.f, 0.f};

    uint32_t left = rounds * cnt, slot = 0;
    for (uint32_t round = 0; round < rounds_all; ++round) {
        if (round < rounds) {
            f32x4_t acc[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < S; ++s)
                if ((uint32_t)s < cnt) {
                    wait_behind<NI>((left < a.ring ? left : a.ring) - 1u);
                    const uint32_t mis = T::BYTES % 16u ? (j * a.rowb + (first_sb + s) * T::BYTES) & 15u : 0u;
                    w.read(slots + slot * SLOT + j * (T::PITCH * 16u), g, mis);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read: the slot may be filled again
                    fetch();
                    --left;
                    if (++slot == a.ring) slot = 0;
                    w.template mul<NF, NV>(x[s], g, acc);
                }
            float* mine = red + (round & 1u) * buf + wave * part;
            if constexpr (!F32) {
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    if (2u * g + v < a.m) mine[(2u * g + v) * 16u + j] = acc[0][v];
            } else {
                const uint32_t per = krows_per(a.m, NF);
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const float last = (acc[f][0] + acc[f][1]) + acc[f][2];  // (columns 12 .. 14)
                    if (g == 3u && per == NV + 1u && f * per + NV < a.m) mine[(f * per + NV) * 16u + j] = last;
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const float s = xor32_add(xor16_add(g < 3u ? acc[f][v] : 0.f));
                        if (g == 0u && (uint32_t)v < per && f * per + v < a.m) mine[(f * per + v) * 16u + j] = s;
                    }
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < 2; ++i) {  // (rows_red <= 2 waves)
            const uint32_t q = wred + i * waves;
            if (q >= rows_red) break;
            const uint32_t org = (q >= a.m) + (q >= 2u * a.m) + (q >= 3u * a.m), row = q - org * a.m, u = (blockIdx.x + (round >> shift) * gridDim.x) * a.rg + org;
            if (u >= a.units) break;
            const float* r = red + (round & 1u) * buf + (org * a.kp * a.m + row) * 16u + j;
            float t[4];
#pragma unroll
            for (uint32_t p = 0; p < 4u; ++p) {
                const float u4 = r[(4u * p + g < a.kp ? 4u * p + g : 0u) * part];
                t[p] = 4u * p + g < a.kp ? u4 : 0.f;
            }
            float v = xor32_add(xor16_add((t[0] + t[1]) + (t[2] + t[3])));
            if constexpr (WHOLE)
                if (__builtin_expect(__any(!(fabsf(v) < __builtin_inff())), 0)) {
                    const float whole = sum_again<TYPE, F32>(row, u, lane, a.swiglu ? round & 1u : 0u);
                    if (!(fabsf(v) < __builtin_inff())) v = whole;
                }
            if (a.swiglu && !(round & 1u)) {
                held[i] = v;
            } else if (g == 0u) {
                uint32_t seg = 0, from = 0;
                if (!a.swiglu)
                    while (seg + 1u < a.nseg && u >= a.end[seg]) from = a.end[seg++];
                const size_t at = (size_t)row * a.n[seg] + (size_t)(u - from) * 16u + j;
                float* y = a.y[seg] + at;
                if (a.swiglu || a.gate)
                    *y = silu_mul_f32(a.swiglu ? held[i] : a.gate[at], v);
                else
                    *y = a.add ? *y + v : v;
            }
        }
    }
}

constexpr size_t kKLds = 160 * 1024 - 512;

template <int TYPE, bool F32, int NV, int NF, int S, int W, bool WHOLE>
int launch_krows(hipStream_t s, KRowsArgs& a, const KSplit& p, uint32_t cus) {
    using T = KWeights<TYPE>;
    constexpr size_t SLOT = 256u * T::PITCH;
    if (!p.kp) return fail(HQ_ERR_UNSUPPORTED, "k rows: %u rows over %u super-blocks", a.m, a.nsb);
    a.kp = p.kp;
    a.rg = p.rg;
    const uint32_t waves = a.kp * a.rg, wgs = (a.units + a.rg - 1u) / a.rg, grid = wgs < cus ? wgs : cus;
    a.base = a.nsb / a.kp;
    a.extra = a.nsb % a.kp;
    a.full = a.units / (grid * a.rg);
    a.rem = a.units % (grid * a.rg);
    const size_t red = 2u * (size_t)waves * a.m * 64u;
    a.ring = (uint32_t)((kKLds - red) / (waves * SLOT));
    a.ring = a.ring < kKMaxRing ? a.ring : kKMaxRing;
    const size_t lds = waves * a.ring * SLOT + red;
    if (waves > (uint32_t)W || a.base + (a.extra ? 1u : 0u) > (uint32_t)S || a.ring < 1u || a.rg * a.m > 2u * waves)
        return fail(HQ_ERR_INVALID_ARGUMENT, "k rows: %u rows, %u super-blocks over %u waves", a.m, a.nsb, waves);
    auto kern = krows_kernel<TYPE, F32, NV, NF, S, W, WHOLE>;
    const size_t ask = lds < 81 * 1024 ? 81 * 1024 : lds;  // one workgroup per CU
    if (int rc = ensure_lds_limit(reinterpret_cast<const void*>(kern), ask, "hipFuncSetAttribute(k rows LDS)")) return rc;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * waves), ask, s, a);
    return check_launch("k rows kernel launch");
}
template <int TYPE, bool F32, int NV, bool WHOLE>
int launch_krows_s(hipStream_t s, KRowsArgs& a, uint32_t cus) {
    const KSplit p = krows_form(TYPE == HQ_Q6_K, F32, a.m, a.nsb, a.units, cus);
    if (p.s == 1u) return launch_krows<TYPE, F32, NV, 1, 1, 16, WHOLE>(s, a, p, cus);
    if constexpr (TYPE != HQ_Q6_K)
        if (p.w == 16u) return launch_krows<TYPE, F32, NV, 1, 2, 16, WHOLE>(s, a, p, cus);
    if (p.s == 2u) return launch_krows<TYPE, F32, NV, 1, 2, 12, WHOLE>(s, a, p, cus);
    return launch_krows<TYPE, F32, NV, 1, 3, 12, WHOLE>(s, a, p, cus);
}
template <int TYPE, bool WHOLE>
int launch_krows_w(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) {
    if (!f32) return launch_krows_s<TYPE, false, 2, WHOLE>(s, a, cus);
    if (a.m <= 4u) return launch_krows_s<TYPE, true, 3, WHOLE>(s, a, cus);  // (nine rows: passes of five and four)
    if (a.m == 5u) return launch_krows_s<TYPE, true, 4, WHOLE>(s, a, cus);
    return launch_krows<TYPE, true, 3, 2, 1, 16, WHOLE>(s, a, krows_form(TYPE == HQ_Q6_K, true, a.m, a.nsb, a.units, cus), cus);
}
template <int TYPE>
int launch_krows_t(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) {
    if constexpr (TYPE == HQ_Q4_0 || TYPE == HQ_Q6_K)
        if (a.whole) return launch_krows_w<TYPE, true>(s, a, f32, cus);
    return launch_krows_w<TYPE, false>(s, a, f32, cus);
}

}  // namespace

// One translation unit per weight type or two.
int launch_krows_q4k(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus);
int launch_krows_q5k(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus);
int launch_krows_q6k(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus);
int launch_krows_q80(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus);
int launch_krows_q40(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus);

}  // namespace hq
