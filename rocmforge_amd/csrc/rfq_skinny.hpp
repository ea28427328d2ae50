// Matrix-core contraction for few rows of activations:  y[m, n] = x[m, k] . dequant(W)[n, k]^T, one launch, no temporary.
//
//   * float32 x, 2..8 rows  (decode batches, rfq_gemv)
//   * float16 a, fewer than 256 rows, arranged ones also more (short prompts, rfq_gemm_f16 / rfq_gemm_f16_arranged)
//
// With so few rows every packed weight byte is wanted once and the matrix cores are nearly idle; what bounds the call is
// the weight stream, the vector instructions that turn codes into operands, and the activations, which every workgroup
// reads whole.  Hence:
//   * The operand of the matrix instruction (v_mfma_f32_16x16x32_f16) is the integer CODE of a weight (exact in fp16) and
//     one instruction covers one 32-element group of 16 weight rows, so a group's scale is applied to its sum in float32:
//     acc += scale * sum.  Weights are never rounded, and a scale may have any float32 value.
//   * Four neighbouring lanes fetch whole 16- or 32-byte pieces of four neighbouring groups of a row (with the lanes of the
//     operand layout, rows side by side, the same loads ran at a quarter of the rate: Q8_0 37 rows 4096 x 4096 16.8 us);
//     the dwords move to the row's operand lanes (ds_bpermute), which trade them with v_permlane32_swap /
//     v_permlane16_swap until each holds its eight codes of every group.  Activations take the same way through LDS.
//   * Mins (Q4_K): the sum of x over a group comes out of the same instruction with a weight operand of ones, already in
//     the layout of the result: acc += min * sum(x).
//   * float32 x is split into two fp16 parts of 11 bits each, hi and 2^11 times what hi leaves, under a power of two per vector
//     and 128-element unit that takes the unit's largest |x| to 2^14 .. 2^15: 23 bits of every x down to 2^-28 of it.  The
//     parts of eight vectors are the sixteen rows of one operand; a unit's sums are float32 and go, times the inverse power,
//     into float64 accumulators, so that neither an outlier nor the length of a row costs a result its precision.
//   * No split of k over workgroups: the wavefronts of a workgroup share 16 * TJ weight rows, take the 128-element units
//     of k in turn and add their results through LDS: one launch, nothing to allocate.
// Measured (cold weights, captured launches; the tiled kernel with its arrangement and its parts -> this one):
//   37 x 4096 -> 4096      Q8_0 33.9 -> 9.8 us    GGUF_Q4_K 26.6 -> 9.2    GGUF_Q6_K 43.5 -> 9.9    Q4_K 22.5 -> 11.3
//   9 x 1024 -> 768        Q8_0 27.9 -> 3.3       GGUF_Q4_K 20.2 -> 3.3    GGUF_Q6_K 36.5 -> 4.0    Q4_K 16.5 -> 4.0
//   48 x 4096 -> 14336     Q8_0 63.8 -> 22.3      GGUF_Q4_K 44.7 -> 21.4   GGUF_Q6_K 82.1 -> 25.1   Q4_K 40.4 -> 31.0
// and decode batches (integer-dot batch kernel, or a launch per vector -> this one):
//   8 x 4096 -> 4096       Q8_0 11.0 -> 8.7 us    GGUF_Q4_K 14.4 -> 8.4    Q6_K 34.1 -> 9.4         MXFP4 33.2 -> 8.7
//   5 x 13824 -> 5120      Q8_0 61 -> 36          GGUF_Q4_K 61 -> 32       GGUF_Q6_K 90 -> 39       Q4_K 73 -> 34
//   error against 64 bits (2-norm of the result), 512 x 13824, 5 vectors: Q6_K 1.07e-7 (float kernel) -> 8.1e-8, Q4_K 1.12e-7 ->
//   7.4e-8, MXFP6 1.02e-7 -> 5.6e-8; (integer-dot kernel) GGUF_Q6_K 2.8e-7 -> 8.0e-8, 8 x 4096 -> 4096 Q8_0 2.7e-7 -> 7.7e-8
// (9.2 us for 37 rows of GGUF_Q4_K is 1 TB/s of weights: what bounds it is vector instructions, 11 per matrix instruction, eight of
// them for scale and min, issued for 59 % of the cycles, and behind them the activations, 384 KB per workgroup through L2 and LDS;
// decode batches issue vector instructions for 40 % of their time and wait for a third of their wavefronts' cycles.)
#pragma once
#include <type_traits>

#include "rfq_code_operands.hpp"

namespace rfq {
namespace skinny {

typedef float v4f_a4 __attribute__((ext_vector_type(4), aligned(4)));

// out[j] in lane (q, i) = in[q] of lane (j, i): a 4 x 4 transposition over the four 16-lane rows.
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b)
{
    const v2u r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b)
{
    const v2u r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
__device__ __forceinline__ void transpose4(uint32_t &a, uint32_t &b, uint32_t &c, uint32_t &d)
{
    swap32(a, c);
    swap32(b, d);
    swap16(a, b);
    swap16(c, d);
}
// every lane's value of group q -> the values of all four groups of its row
__device__ __forceinline__ void spread4(float v, float (&out)[4])
{
    uint32_t a = __float_as_uint(v), b = a, c = a, d = a;
    transpose4(a, b, c, d);
    out[0] = __uint_as_float(a); out[1] = __uint_as_float(b); out[2] = __uint_as_float(c); out[3] = __uint_as_float(d);
}

__device__ __forceinline__ void spread4u(uint32_t v, uint32_t (&out)[4])
{
    out[0] = out[1] = out[2] = out[3] = v;
    transpose4(out[0], out[1], out[2], out[3]);
}

// the eight nibbles of a dword in their order, as fp16 pairs of nibble + bias
__device__ __forceinline__ v4u nibbles_in_order(uint32_t d, float bias)
{
    const uint32_t even = d & 0x0F0F0F0Fu, odd = (d >> 4) & 0x0F0F0F0Fu;
    v4u o;
    uint32_t a, b;
    bytes2h(__builtin_amdgcn_perm(odd, even, 0x05010400u), bias, a, b);
    o[0] = a; o[1] = b;
    bytes2h(__builtin_amdgcn_perm(odd, even, 0x07030602u), bias, a, b);
    o[2] = a; o[3] = b;
    return o;
}
// (any address: where a format's blocks are fetched through aligned windows the caller has rounded it down)
template <int NW> __device__ __forceinline__ void load_dwords(const uint8_t *a, uint32_t (&d)[NW])
{
    typedef uint32_t v4a1 __attribute__((ext_vector_type(4), aligned(1)));
    typedef uint32_t v2a1 __attribute__((ext_vector_type(2), aligned(1)));
    int i = 0;
#pragma unroll
    for (; i + 4 <= NW; i += 4) {
        const v4a1 v = *reinterpret_cast<const v4a1 *>(a + 4 * i);
        d[i] = v[0]; d[i + 1] = v[1]; d[i + 2] = v[2]; d[i + 3] = v[3];
    }
    if (i + 2 <= NW) {
        const v2a1 v = *reinterpret_cast<const v2a1 *>(a + 4 * i);
        d[i] = v[0]; d[i + 1] = v[1];
        i += 2;
    }
    if (i < NW) d[i] = ld<uint32_t>(a + 4 * i);
}
// Which eight elements of a group lane row q holds, and in which order its four operand dwords hold them.
enum { OCTET, OCTET_SWAPPED, HALVES };                           // 8q..  |  8q'.. (q' = q with its bits swapped)  |  4q.. and 16+4q..
enum { P04, P01, P02, P26 };                                     // (0,4)(1,5)(2,6)(3,7) | (0,1)(2,3)(4,5)(6,7) | (0,2)(1,3)(4,6)(5,7) | (0,2)(4,6)(1,3)(5,7)

// The matrix instruction gives the same bits whatever order the eight k of a lane have, as long as both operands have the same.  So
// the float16 kernel leaves the activations as they come (P01 from rows, P04 arranged) and turn<TO>() and frag_as<TO>() bring the
// codes into that order: a few instructions per unit of W where turning the activations took four per operand and group.
// W<FMT>: load() fetches the dwords r[] that lane 4 * i + g holds of group g of the 128-element unit `u` of row i (four
// neighbouring lanes on neighbouring bytes: a load whose neighbouring lanes sit in different rows runs at a quarter of the
// rate).  The dwords then move to lane 16 * g + i; open() turns them into codes and scales there (dead: the group lies past
// the end of the row and its weights count as zero), frag(j) gives the operand of group j, sc(j, half) / mn(j) its scale
// and min.
template <int FMT> struct W;

template <> struct W<RFQ_Q4_0> {
    static constexpr int ORDER = OCTET, PAIRS = P04, NR = 5;
    static constexpr bool MINS = false, SPLIT16 = false;
    uint32_t r[NR], q[4];
    float sc4[4];
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g) { load_dwords<5>(row + (uint32_t)(4 * u + g) * 20u, r); }
    __device__ __forceinline__ void open(int, bool dead)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = r[i + 1];
        transpose4(q[0], q[1], q[2], q[3]);
        spread4(dead ? 0.f : __uint_as_float(r[0]), sc4);
    }
    __device__ __forceinline__ v4u frag(int j) const { return v4u{nib2h<0>(q[j], -8.f), nib2h<4>(q[j], -8.f), nib2h<8>(q[j], -8.f), nib2h<12>(q[j], -8.f)}; }
    template <int TO> __device__ __forceinline__ void turn() {}
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const
    {
        if constexpr (TO == P04) return frag(j);
        else return nibbles_in_order(q[j], -8.f);
    }
    __device__ __forceinline__ float sc(int j, int) const { return sc4[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};

// The GGUF blocks start on multiples of 2: the aligned dwords that hold the block are fetched (each holds a byte of it),
// and the block's byte offset in the first (0 or 2) travels along.
template <> struct W<RFQ_GGUF_Q4_0> {
    static constexpr int ORDER = HALVES, PAIRS = P02, NR = 6;
    static constexpr bool MINS = false, SPLIT16 = false;
    uint32_t r[NR], q[4];
    float sc4[4];
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *p = row + (uint32_t)(4 * u + g) * 18u;
        const uint32_t o = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3u);
        uint32_t v[5];
        load_dwords<5>(p - o, v);
#pragma unroll
        for (int i = 0; i < 5; i++) r[i] = v[i];
        r[5] = o;
    }
    __device__ __forceinline__ void open(int, bool dead)
    {
        const uint32_t sel = 0x05040302u + __builtin_amdgcn_perm(0u, r[5], 0u);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel);
        transpose4(q[0], q[1], q[2], q[3]);
        spread4(dead ? 0.f : f16_bits_to_f32((uint16_t)(r[0] >> (8u * r[5]))), sc4);
    }
    __device__ __forceinline__ v4u frag(int j) const { return v4u{nib2h<0>(q[j], -8.f), nib2h<8>(q[j], -8.f), nib2h<4>(q[j], -8.f), nib2h<12>(q[j], -8.f)}; }
    template <int TO> __device__ __forceinline__ void turn()
    {
        if constexpr (TO == P01) {
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_perm(0u, q[i], 0x03010200u);
        }
    }
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const { return frag(j); }
    __device__ __forceinline__ float sc(int j, int) const { return sc4[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};

template <int FMT> struct W8 {                                   // Q8_0 (f32 scale, byte - 128), GGUF_Q8_0 (f16 scale, int8)
    static constexpr int ORDER = OCTET, PAIRS = P01, NR = FMT == RFQ_Q8_0 ? 9 : 10;
    static constexpr bool MINS = false, SPLIT16 = false;
    uint32_t r[NR], q[8];
    float sc4[4];
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *p = row + (uint32_t)(4 * u + g) * (FMT == RFQ_Q8_0 ? 36u : 34u);
        const uint32_t o = FMT == RFQ_Q8_0 ? 0u : (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3u);
        uint32_t v[9];
        load_dwords<9>(p - o, v);
#pragma unroll
        for (int i = 0; i < 9; i++) r[i] = v[i];
        if constexpr (FMT != RFQ_Q8_0) r[9] = o;
    }
    __device__ __forceinline__ void open(int, bool dead)
    {
        if constexpr (FMT == RFQ_Q8_0) {
#pragma unroll
            for (int i = 0; i < 8; i++) q[i] = r[i + 1];
            spread4(dead ? 0.f : __uint_as_float(r[0]), sc4);
        } else {
            const uint32_t sel = 0x05040302u + __builtin_amdgcn_perm(0u, r[9], 0u);
#pragma unroll
            for (int i = 0; i < 8; i++) q[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel) ^ 0x80808080u;
            spread4(dead ? 0.f : f16_bits_to_f32((uint16_t)(r[0] >> (8u * r[9]))), sc4);
        }
        transpose4(q[0], q[2], q[4], q[6]);                       // dword pairs: lane row q gets bytes 8q .. 8q + 7 of group j
        transpose4(q[1], q[3], q[5], q[7]);
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        uint32_t a, b, c, d;
        bytes2h(q[2 * j], -128.f, a, b);
        bytes2h(q[2 * j + 1], -128.f, c, d);
        return v4u{a, b, c, d};
    }
    template <int TO> __device__ __forceinline__ void turn()
    {
        if constexpr (TO == P04) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t a = q[2 * j], b = q[2 * j + 1];
                q[2 * j] = __builtin_amdgcn_perm(b, a, 0x05010400u);
                q[2 * j + 1] = __builtin_amdgcn_perm(b, a, 0x07030602u);
            }
        }
    }
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const { return frag(j); }
    __device__ __forceinline__ float sc(int j, int) const { return sc4[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};
template <> struct W<RFQ_Q8_0> : W8<RFQ_Q8_0> {};
template <> struct W<RFQ_GGUF_Q8_0> : W8<RFQ_GGUF_Q8_0> {};

// What the four lanes of a row share (scales, mins) is fetched as one dword per lane and spread: one load and one move to the
// operand lanes instead of three or four of each.
template <> struct W<RFQ_Q4_K> {                                 // 256-byte layout: 8 f16 scales, 8 i8 mins, nibbles at 32 + 28 * sb
    static constexpr int ORDER = OCTET, PAIRS = P04, NR = 5;
    static constexpr bool MINS = true, SPLIT16 = false;
    struct U4 { uint32_t v[4]; };
    uint32_t r[NR], q[4], hd[4];
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 256u;
        const int h = u & 1;
        // (lanes 0, 1: two scales each; lanes 2, 3: the unit's four mins)
        r[4] = ld<uint32_t>(blk + (g < 2 ? 8 * h + 4 * g : 16 + 4 * h));
        const U4 v = ld_once<U4>(blk + 32 + 28 * (4 * h + g));
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = v.v[i];
    }
    __device__ __forceinline__ void open(int, bool)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = r[i];
        transpose4(q[0], q[1], q[2], q[3]);
        spread4u(r[4], hd);
    }
    __device__ __forceinline__ v4u frag(int j) const { return v4u{nib2h<0>(q[j], 0.f), nib2h<4>(q[j], 0.f), nib2h<8>(q[j], 0.f), nib2h<12>(q[j], 0.f)}; }
    template <int TO> __device__ __forceinline__ void turn() {}
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const
    {
        if constexpr (TO == P04) return frag(j);
        else return nibbles_in_order(q[j], 0.f);
    }
    __device__ __forceinline__ float sc(int j, int) const { return f16_bits_to_f32((uint16_t)(hd[j >> 1] >> (16 * (j & 1)))); }
    __device__ __forceinline__ float mn(int j) const { return (float)(int)(int8_t)(hd[2] >> (8 * j)); }
};

template <> struct W<RFQ_GGUF_Q4_K> {
    static constexpr int ORDER = OCTET_SWAPPED, PAIRS = P02, NR = 5;
    static constexpr bool MINS = true, SPLIT16 = false;
    uint32_t r[NR], q[4];
    uint32_t scb, mnb; float d, dm;
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 144u;
        uint32_t b[4];
        r[4] = ld<uint32_t>(blk + 4 * g);
        load_dwords<4>(blk + 16 + 64 * (u & 1) + 16 * g, b);
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = b[i];
    }
    // lane row (q1 q0) holds bytes 16 q0 .. of the unit's 64-element chunk q1; it keeps bytes 16 q0 + 8 q1 .. +8 of both
    __device__ __forceinline__ void open(int u, bool)
    {
        uint32_t hd[4];
        spread4u(r[4], hd);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = r[i];
        swap32(q[0], q[2]);
        swap32(q[1], q[3]);
        if ((u & 1) == 0) {
            scb = hd[1] & 0x3F3F3F3Fu;
            mnb = hd[2] & 0x3F3F3F3Fu;
        } else {
            scb = (hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u);
            mnb = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
        }
        d = f16_bits_to_f32((uint16_t)hd[0]);
        dm = -f16_bits_to_f32((uint16_t)(hd[0] >> 16));
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        const uint32_t a = q[2 * (j >> 1)], b = q[2 * (j >> 1) + 1];
        if (j & 1) return v4u{nib2h<4>(a, 0.f), nib2h<12>(a, 0.f), nib2h<4>(b, 0.f), nib2h<12>(b, 0.f)};
        return v4u{nib2h<0>(a, 0.f), nib2h<8>(a, 0.f), nib2h<0>(b, 0.f), nib2h<8>(b, 0.f)};
    }
    template <int TO> __device__ __forceinline__ void turn()
    {
        if constexpr (TO == P01) {
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_perm(0u, q[i], 0x03010200u);
        } else if constexpr (TO == P04) {
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                const uint32_t a = q[i], b = q[i + 1];
                q[i] = __builtin_amdgcn_perm(b, a, 0x05040100u);
                q[i + 1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
            }
        }
    }
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const { return frag(j); }
    __device__ __forceinline__ float sc(int j, int) const { return d * (float)((scb >> (8 * j)) & 255u); }
    __device__ __forceinline__ float mn(int j) const { return dm * (float)((mnb >> (8 * j)) & 255u); }
};

// Scales per 16 elements: a group's operand is two halves of 16, each with an instruction (16x16x16) of its own.
template <> struct W<RFQ_Q6_K> {
    static constexpr int ORDER = HALVES, PAIRS = P01, NR = 7;
    static constexpr bool MINS = false, SPLIT16 = true;
    uint32_t r[NR];
    uint32_t q[8]; float sa[4], sb[4];
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 256u;
        const int c = 4 * (u & 1) + g;
        r[6] = ld<uint32_t>(blk + 4 * c);
        uint32_t v[6];
        load_dwords<6>(blk + 32 + 24 * c, v);
#pragma unroll
        for (int i = 0; i < 6; i++) r[i] = v[i];
    }
    static __device__ __forceinline__ uint32_t bytes_of(uint32_t t)  // four 6-bit codes in bits 0..23 -> four bytes of code ^ 32
    {
        uint32_t v = t;
        asm("v_lshrrev_b32_sdwa %0, %2, %1 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(v) : "v"(t), "i"(6));
        asm("v_lshrrev_b32_sdwa %0, %2, %1 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(v) : "v"(t), "i"(12));
        asm("v_lshrrev_b32_sdwa %0, %2, %1 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(v) : "v"(t), "i"(18));
        return (v & 0x3F3F3F3Fu) ^ 0x20202020u;
    }
    __device__ __forceinline__ void open(int, bool)
    {
#pragma unroll
        for (int g = 0; g < 8; g++) {
            const int b = 3 * (g & 3), d = 3 * (g >> 2);
            const uint32_t t = b == 0 ? r[d] : b == 9 ? r[d + 2] >> 8 : __builtin_amdgcn_alignbit(r[d + b / 4 + 1], r[d + b / 4], 8 * (b & 3));
            q[g] = bytes_of(t);
        }
        transpose4(q[0], q[1], q[2], q[3]);                       // q[j] / q[4 + j]: this lane row's four codes of group j's halves
        transpose4(q[4], q[5], q[6], q[7]);
        spread4(f16_bits_to_f32((uint16_t)r[6]), sa);
        spread4(f16_bits_to_f32((uint16_t)(r[6] >> 16)), sb);
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        uint32_t a, b, c, d;
        bytes2h(q[j], -32.f, a, b);
        bytes2h(q[4 + j], -32.f, c, d);
        return v4u{a, b, c, d};
    }
    template <int TO> __device__ __forceinline__ void turn() {}
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const { return frag(j); }
    __device__ __forceinline__ float sc(int j, int h) const { return h ? sb[j] : sa[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};

template <> struct W<RFQ_GGUF_Q6_K> {
    static constexpr int ORDER = HALVES, PAIRS = P01, NR = 10;
    static constexpr bool MINS = false, SPLIT16 = true;
    uint32_t r[NR];
    uint32_t q[4], c[2], s[2]; float d;
    // Blocks start on multiples of 2 and every piece on a multiple of 4 from there: the aligned dwords around a piece, o (0
    // or 2) bytes before it; the last is read only where it holds a byte of the piece.
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 210u;
        const int half = u & 1, gs = ((g & 1) << 1) | (g >> 1);
        const uint32_t o = (uint32_t)(reinterpret_cast<uintptr_t>(blk) & 3u);
        const uint8_t *a = blk - o;
        uint32_t v[4], t[2];
        load_dwords<4>(a + 64 * half + 16 * g, v);                // lower nibbles: 16 of the unit's 64 bytes
        r[4] = *reinterpret_cast<const uint32_t *>(a + 64 * half + 16 * g + (o ? 16 : 12));
        load_dwords<2>(a + 128 + 32 * half + 8 * gs, t);          // upper bit pairs: 8 of its 32 bytes
        r[7] = *reinterpret_cast<const uint32_t *>(a + 128 + 32 * half + 8 * gs + (o ? 8 : 4));
        // lanes 0 .. 2: the dwords of its eight scales, lane 3: d
        r[8] = *reinterpret_cast<const uint32_t *>(a + (g == 3 ? 208 : 192 + 8 * half + (g == 2 && !o ? 4 : 4 * g)));
        r[9] = o;
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = v[i];
        r[5] = t[0]; r[6] = t[1];
    }
    // Lower nibbles: lane row (q1 q0) holds bytes 16 q0 .. of part q1 (groups with even / odd number); two exchanges give every
    // lane row dword q of both halves of both parts.  Bit pairs: lane row (q1 q0) holds dwords 4 q0 + 2 q1, + 1 of eight; one
    // exchange gives it dword q of both halves.
    __device__ __forceinline__ void open(int, bool)
    {
        const uint32_t sel = 0x03020100u + __builtin_amdgcn_perm(0u, r[9], 0u);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel);
#pragma unroll
        for (int i = 0; i < 2; i++) c[i] = __builtin_amdgcn_perm(r[i + 6], r[i + 5], sel);
        swap32(q[0], q[2]);
        swap32(q[1], q[3]);
        swap16(q[0], q[1]);
        swap16(q[2], q[3]);
        swap16(c[0], c[1]);
        uint32_t hd[4];
        spread4u(r[8], hd);
        s[0] = __builtin_amdgcn_perm(hd[1], hd[0], sel);
        s[1] = __builtin_amdgcn_perm(hd[2], hd[1], sel);
        d = f16_bits_to_f32((uint16_t)(hd[3] >> (8u * r[9])));
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        v4u o;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const uint32_t l = (q[2 * (j & 1) + e] >> (4 * (j >> 1))) & 0x0F0F0F0Fu;
            const uint32_t t = (j < 2 ? c[e] << (4 - 2 * j) : c[e] >> (2 * j - 4)) & 0x30303030u;
            uint32_t p, r2;
            bytes2h(l | t, -32.f, p, r2);
            o[2 * e] = p;
            o[2 * e + 1] = r2;
        }
        return o;
    }
    template <int TO> __device__ __forceinline__ void turn() {}
    template <int TO> __device__ __forceinline__ v4u frag_as(int j) const { return frag(j); }
    __device__ __forceinline__ float sc(int j, int hf) const { const int at = 2 * j + hf; return d * (float)(int)(int8_t)(s[at >> 2] >> (8 * (at & 3))); }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};

// The MXFP formats: the operand is the decoded code (MxfpBlock::decode_e2m1 / decode_e2m3, src/loader/mxfp.rs:234-293), a
// multiple of 1/16 below 8 and exact in fp16.  The reference clamps value * 2^e to +-BOUND (mxfp.rs:196-203), which moves a
// value only for e >= 1, and from e = 5 on every value but 0 sits at the bound: a wavefront that holds such a block (one
// ballot) multiplies the block's operand by 2^min(e, 5), clamps it and gives the block the scale 1.
template <int FMT> struct WMx {
    static constexpr int ND = FMT == RFQ_MXFP4 ? 4 : 6;           // dwords of codes behind the exponent byte
    static constexpr int ORDER = OCTET, PAIRS = FMT == RFQ_MXFP4 ? P26 : P01, NR = ND + 2;
    static constexpr bool MINS = false, SPLIT16 = false;
    uint32_t r[NR], q[8];
    float sc4[4], up4[4];
    bool clamp;
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *p = row + (uint32_t)(4 * u + g) * (uint32_t)(1 + 4 * ND);
        const uint32_t o = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3u);
        uint32_t v[ND + 1];
        load_dwords<ND + 1>(p - o, v);                            // (o + 1 + 4 ND <= 4 (ND + 1): each holds a byte of the block)
#pragma unroll
        for (int i = 0; i <= ND; i++) r[i] = v[i];
        r[ND + 1] = o;
    }
    __device__ __forceinline__ void open(int, bool dead)
    {
        const uint32_t sel = 0x04030201u + __builtin_amdgcn_perm(0u, r[ND + 1], 0u);
        uint32_t c[ND];
#pragma unroll
        for (int i = 0; i < ND; i++) c[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel);
        const int e = (int)(int8_t)(r[0] >> (8u * r[ND + 1]));
        clamp = __builtin_amdgcn_ballot_w64(e >= 1) != 0;
        spread4(dead ? 0.f : e >= 1 ? 1.0f : mx_scale(e), sc4);
        if (clamp) spread4(e >= 1 ? mx_scale(e < 5 ? e : 5) : 1.0f, up4);
        if constexpr (FMT == RFQ_MXFP4) {
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = c[i];
            transpose4(q[0], q[1], q[2], q[3]);
        } else {
            // elements 4j .. 4j+3 at bits 10, 4, 14 and 24 of the 32 bits from bit 24 j (element 31 is never written: code 0)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int d = 24 * j / 32, sh = 24 * j % 32;
                const uint32_t w = sh == 0 ? c[d] : __builtin_amdgcn_alignbit(d + 1 < ND ? c[d + 1] : 0u, c[d], sh);
                q[j] = ((w >> 10) & 0x3Fu) | ((w << 4) & 0x3F00u) | ((w << 2) & 0x3F0000u) | (j < 7 ? w & 0x3F000000u : 0u);
            }
            transpose4(q[0], q[2], q[4], q[6]);
            transpose4(q[1], q[3], q[5], q[7]);
        }
    }
    // four E2M1 codes (one per byte) -> the high bytes of their fp16 values (the low bytes are zero)
    static __device__ __forceinline__ uint32_t e2m1(uint32_t c)
    {
        const uint32_t at = c & 0x07070707u, s = (c >> 3) & 0x01010101u, neg = (s << 8) - s;
        const uint32_t pos = __builtin_amdgcn_perm(0x48444440u, 0x403C3C00u, at), mns = __builtin_amdgcn_perm(0xC8C4C4C0u, 0xC0BCBCB8u, at);
        return (neg & mns) | (~neg & pos);
    }
    // two E2M3 codes in the 16-bit halves -> fp16: 0x3800 + (code & 31) * 128 is (1 + m / 8) * 2^(x - 1); code 0 is zero
    static __device__ __forceinline__ uint32_t e2m3(uint32_t p)
    {
        typedef uint16_t v2s __attribute__((ext_vector_type(2)));
        const uint32_t h = (((p & 0x001F001Fu) << 7) + 0x38003800u) | ((p & 0x00200020u) << 10);
        v2s a, b;
        __builtin_memcpy(&a, &p, 4);
        __builtin_memcpy(&b, &h, 4);
        a = __builtin_elementwise_min(a, v2s{1, 1}) * b;
        uint32_t o;
        __builtin_memcpy(&o, &a, 4);
        return o;
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        v4u o;
        if constexpr (FMT == RFQ_MXFP4) {                         // element 2 b of an octet is the high nibble of byte b
            const uint32_t ev = e2m1((q[j] >> 4) & 0x0F0F0F0Fu), od = e2m1(q[j] & 0x0F0F0F0Fu);
            o = v4u{__builtin_amdgcn_perm(ev, ev, 0x010C000Cu), __builtin_amdgcn_perm(ev, ev, 0x030C020Cu),
                    __builtin_amdgcn_perm(od, od, 0x010C000Cu), __builtin_amdgcn_perm(od, od, 0x030C020Cu)};
        } else {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                o[2 * e] = e2m3(__builtin_amdgcn_perm(0u, q[2 * j + e], 0x0C010C00u));
                o[2 * e + 1] = e2m3(__builtin_amdgcn_perm(0u, q[2 * j + e], 0x0C030C02u));
            }
        }
        if (clamp) {
            const _Float16 up = (_Float16)up4[j], bound = FMT == RFQ_MXFP4 ? (_Float16)8.0f : (_Float16)7.5f;
            const v2h lim = {bound, bound};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v2h h;
                const uint32_t bits = o[i];
                __builtin_memcpy(&h, &bits, 4);
                h = __builtin_elementwise_max(__builtin_elementwise_min(h * v2h{up, up}, lim), -lim);
                uint32_t t;
                __builtin_memcpy(&t, &h, 4);
                o[i] = t;
            }
        }
        return o;
    }
    __device__ __forceinline__ float sc(int j, int) const { return sc4[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};
template <> struct W<RFQ_MXFP4> : WMx<RFQ_MXFP4> {};
template <> struct W<RFQ_MXFP6_E2M3> : WMx<RFQ_MXFP6_E2M3> {};

// r[] of lane 4 * i + g -> lane 16 * g + i
template <int FMT> __device__ __forceinline__ W<FMT> placed(const W<FMT> &raw, int from4)
{
    W<FMT> o;
#pragma unroll
    for (int d = 0; d < W<FMT>::NR; d++) o.r[d] = (uint32_t)__builtin_amdgcn_ds_bpermute(from4, (int)raw.r[d]);
    return o;
}

__device__ __forceinline__ int row_part(int order, int q)         // the number of the octet / quarter-half of lane row q
{
    return order == OCTET_SWAPPED ? ((q & 1) << 1) | (q >> 1) : q;
}

template <int PAIRS> __device__ __forceinline__ constexpr int pair_of(int r, int h)  // element h of operand dword r
{
    return PAIRS == P04 ? r + 4 * h : PAIRS == P01 ? 2 * r + h : PAIRS == P02 ? (r >> 1) * 4 + (r & 1) + 2 * h : (r & 1) * 4 + (r >> 1) + 2 * h;
}

template <bool SPLIT16>
__device__ __forceinline__ void contract(const v4u &xa, const v4u &wf, v4f (&d)[2])
{
    if constexpr (SPLIT16) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const v2u x2 = {xa[2 * h], xa[2 * h + 1]}, w2 = {wf[2 * h], wf[2 * h + 1]};
            v4h x4, w4;
            __builtin_memcpy(&x4, &x2, 8);
            __builtin_memcpy(&w4, &w2, 8);
            d[h] = __builtin_amdgcn_mfma_f32_16x16x16f16(x4, w4, d[h], 0, 0, 0);
        }
    } else {
        v8h x8, w8;
        __builtin_memcpy(&x8, &xa, 16);
        __builtin_memcpy(&w8, &wf, 16);
        d[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x8, w8, d[0], 0, 0, 0);
    }
}

// Between a wavefront's writes to its own part of LDS and other lanes' reads of them (and before the part is written again):
// the hardware completes a wavefront's LDS operations in order, this keeps the compiler from moving them across.  No instruction.
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- float32 x, m <= 8 -----------------------------------------------------------------------------------------------
// blockDim = 64 * waves.  w2 != nullptr (TJ even): the odd row tiles come from w2, a second matrix of the same shape (gate and
// up projections), and y[j] = swiglu(row j of w, row j of w2) as the reference defines it (kernels/swiglu.hip:40-62).  NORM:
// x is RMSNorm(x) * norm_w (kernels/rms_norm.hip:40-84): x * norm_w is multiplied and the vector's factor
// 1 / sqrt(mean(x^2) + eps) applied to its results.
// LDS: per wavefront x_bytes for its unit of x as fp16 parts (plane hi, plane lo; vector; operand
// order), later the wavefronts' results.
// x goes global -> registers (sixteen lanes per vector, eight elements each: consecutive lanes on consecutive bytes) ->
// two fp16 parts -> LDS -> operands: every element is converted once per workgroup and unit.
constexpr int XROW = 256 + 16;                                    // bytes of a vector's 128 elements, bank-skewed
// (the two parts of MV vectors as rows of the operand, and the vectors' inverse scales)
template <int MV> constexpr int x_bytes() { return 2 * MV * XROW + MV * 4; }
template <int TJ, int MV> constexpr int gemv_lds(int waves)
{
    // (the results are followed by the vectors' sums of squares, MV per wavefront, or of prepared x MV in double: x_bytes leaves room)
    static_assert(x_bytes<MV>() >= MV * 16 * TJ * 4 + MV * 8, "room for the sums of squares");
    return waves * (x_bytes<MV>() > MV * (16 * TJ + 1) * 4 ? x_bytes<MV>() : MV * (16 * TJ + 1) * 4);
}

// The largest magnitude (fmaxf of fabsf spends an instruction more per operand on signalling NaNs).
__device__ __forceinline__ float max3_abs(float a, float b, float c)
{
    float o;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(o) : "v"(a), "v"(b), "v"(c));
    return o;
}

// The largest of the sixteen lanes of a lane row, in all of them.
__device__ __forceinline__ uint32_t max16(uint32_t v)
{
    auto step = [&](auto ctrl) {
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xF, 0xF, true);
        v = v > o ? v : o;
    };
    step(std::integral_constant<int, 0xB1>{});                    // quad_perm [1 0 3 2]
    step(std::integral_constant<int, 0x4E>{});                    // quad_perm [2 3 0 1]
    step(std::integral_constant<int, 0x141>{});                   // row_half_mirror
    step(std::integral_constant<int, 0x140>{});                   // row_mirror
    return v;
}

// The power of two that takes a vector's largest |x| in a unit (ex: its biased exponent) to 2^top .. 2^(top + 1), and its inverse.
template <bool LOW> __device__ __forceinline__ void octet_scale(int ex, int top, float &s, float &inv)
{
    int se = 254 + top - ex;                                      // s = 2^(top - (ex - 127))
    se = se > 243 ? 243 : LOW && se < 1 ? 1 : se;                 // (2048 s stays finite, s above zero)
    s = __uint_as_float((uint32_t)se << 23);
    inv = __uint_as_float((uint32_t)(254 - se) << 23);
}
// Octet e (8 consecutive elements of one vector) under that power of two as the two fp16 parts.
template <int PAIRS>
__device__ __forceinline__ void split_octet(const float (&e)[8], float s, float inv, uint32_t (&hi)[4], uint32_t (&lo)[4])
{
#pragma unroll
    for (int r = 0; r < 4; r++) {
        // (x * s, x - hi / s and its multiple by 2048 s are exact: a part is rounded once, to fp16)
        const float a = e[pair_of<PAIRS>(r, 0)], b = e[pair_of<PAIRS>(r, 1)];
        v2h h = {(_Float16)__builtin_fmaf(a, s, 0.0f), (_Float16)__builtin_fmaf(b, s, 0.0f)};
        __builtin_memcpy(&hi[r], &h, 4);
        asm("" : "+v"(hi[r]));                                    // (one conversion of each product, not one per use)
        __builtin_memcpy(&h, &hi[r], 4);
        const float ra = __builtin_fmaf((float)h[0], -inv, a), rb = __builtin_fmaf((float)h[1], -inv, b);
        const v2h l = {(_Float16)__builtin_fmaf(ra, s * 2048.0f, 0.0f), (_Float16)__builtin_fmaf(rb, s * 2048.0f, 0.0f)};
        __builtin_memcpy(&lo[r], &l, 4);
    }
}
// What an infinity leaves as its lower part is a NaN, and with it every result of the vector; without it the infinity's product
// with a weight that is not zero stays one.
__device__ __forceinline__ uint32_t without_infinities(uint32_t hi, uint32_t lo)
{
    return lo & (((hi & 0x7FFFu) == 0x7C00u ? 0u : 0xFFFFu) | ((hi & 0x7FFF0000u) == 0x7C000000u ? 0u : 0xFFFF0000u));
}

// x prepared for several workgroups (SkinnyGemv::ready), in the caller's scratch memory: per unit, group and lane row the operands
// of the m vectors' upper parts and then of their lower parts, 16 bytes each; behind all units, eight floats per unit
// each, the vectors' inverse scales and (norm) their sums of squares.
__host__ __device__ constexpr size_t ready_squares(int m, int units) { return (size_t)units * (512 * m + 32); }

template <int ORDER, int PAIRS>
__global__ void __launch_bounds__(128)
prepare_x_kernel(const float *__restrict__ x, const float *__restrict__ norm_w, int m, int k, uint8_t *__restrict__ out, int keep_infinities)
{
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4, u = blockIdx.x, units = gridDim.x;
    const int v = 4 * (int)(threadIdx.x >> 6) + q, at = 128 * u + 8 * i;
    float e[8], ss = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; c++) e[c] = 0.0f;
    if (at < k) {
        const float *p = x + (size_t)(v < m ? v : m - 1) * k + at;
        const v4f a = *reinterpret_cast<const v4f_a4 *>(p), b = *reinterpret_cast<const v4f_a4 *>(p + 4);
#pragma unroll
        for (int c = 0; c < 4; c++) { e[c] = a[c]; e[4 + c] = b[c]; }
        if (norm_w != nullptr) {
            const v4f na = *reinterpret_cast<const v4f *>(norm_w + at), nb = *reinterpret_cast<const v4f *>(norm_w + at + 4);
#pragma unroll
            for (int c = 0; c < 8; c++) {
                ss = __builtin_fmaf(e[c], e[c], ss);
                e[c] *= c < 4 ? na[c & 3] : nb[c & 3];
            }
        }
    }
    const float mx = max3_abs(max3_abs(e[0], e[1], e[2]), max3_abs(e[3], e[4], e[5]), max3_abs(e[6], e[7], 0.0f));
    const int ex = (int)(max16(__float_as_uint(mx)) >> 23);
    uint32_t hi[4], lo[4];
    float s, inv;
    octet_scale<false>(ex, 14, s, inv);
    split_octet<PAIRS>(e, s, inv, hi, lo);
    if (keep_infinities && ex == 255) {
#pragma unroll
        for (int r = 0; r < 4; r++) lo[r] = without_infinities(hi[r], lo[r]);
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) ss += __shfl_xor(ss, o);
    if (v >= m) return;
    uint8_t *const unit = out + (size_t)u * (512 * m);
    const int o = i & 3, j4 = (i >> 2) * 4;                       // octet o of group i >> 2
    if constexpr (ORDER <= OCTET_SWAPPED) {
        uint8_t *const to = unit + ((j4 + row_part(ORDER, o)) * (2 * m) + v) * 16;
        *reinterpret_cast<v4u *>(to) = v4u{hi[0], hi[1], hi[2], hi[3]};
        *reinterpret_cast<v4u *>(to + m * 16) = v4u{lo[0], lo[1], lo[2], lo[3]};
    } else {
        uint8_t *const t0 = unit + ((j4 + 2 * (o & 1)) * (2 * m) + v) * 16 + (o >> 1) * 8, *const t1 = t0 + 2 * m * 16;
        *reinterpret_cast<v2u *>(t0) = v2u{hi[0], hi[1]};
        *reinterpret_cast<v2u *>(t0 + m * 16) = v2u{lo[0], lo[1]};
        *reinterpret_cast<v2u *>(t1) = v2u{hi[2], hi[3]};
        *reinterpret_cast<v2u *>(t1 + m * 16) = v2u{lo[2], lo[3]};
    }
    if (i == 0) {
        reinterpret_cast<float *>(out + (size_t)units * (512 * m))[u * 8 + v] = inv;
        reinterpret_cast<float *>(out + ready_squares(m, units))[u * 8 + v] = ss;
    }
}

// MV: 4 or 8 vectors, m <= MV.  READY: x comes prepared (prepare_x_kernel) and no workgroup converts it.
template <int FMT, int TJ, int MV, int D, int WAVES, bool NORM, bool READY>
__global__ void __launch_bounds__(64 * WAVES, (FMT == RFQ_MXFP4 && TJ == 2 && MV == 4 && !NORM ? 4 : 1))   // (128 registers, which it misses by two: two workgroups per CU)
gemv_skinny_kernel(const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y, int m, int n, int k,
                   const uint8_t *__restrict__ w2, const float *__restrict__ norm_w, float eps, int keep_infinities, const uint8_t *__restrict__ ready)
{
    typedef W<FMT> WF;
    constexpr int P = MV / 4;                                     // octets of x per lane and unit
    // With one row tile a unit's x is taken and its scale found (a chain of nine instructions) beside the sums of the unit
    // before (GGUF_Q4_0 5 x 14336 -> 4096 22.2 -> 19.8 us); with more, the registers it needs would leave room for one
    // workgroup per CU instead of two, or spill (GGUF_Q6_K 5 x 4096 -> 14336 28 -> 76 us).
    constexpr bool AHEAD = TJ == 1 && !READY;
    // (e and xr then both go round the loop.  Left free, the compiler gives these forms' e the registers of xr, fetches into others and
    // waits at once to move them: GGUF_Q4_0 4 x 4096 -> 4096 and MXFP4 lost 3 to 5 %)
    constexpr bool MOVED = AHEAD && !NORM && MV == 4 && (FMT == RFQ_Q4_0 || FMT == RFQ_GGUF_Q4_0 || FMT == RFQ_MXFP4 || FMT == RFQ_MXFP6_E2M3);
    constexpr bool F32_SCALE = FMT == RFQ_Q4_0 || FMT == RFQ_Q8_0;
    constexpr bool INFINITIES = FMT == RFQ_Q4_K || FMT == RFQ_Q6_K || FMT == RFQ_MXFP4 || FMT == RFQ_MXFP6_E2M3;   // (see keeps_infinities)
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int groups = k >> 5, units = (groups + 3) >> 2;
    const bool glu = TJ >= 2 && w2 != nullptr;
    const int n0 = blockIdx.x * (glu ? 8 * TJ : 16 * TJ);
    const size_t row_bytes = (size_t)(k / Fmt<FMT>::BE) * Fmt<FMT>::BB;
    const uint8_t *row[TJ];                                       // (weights: lane 4 * i + g fetches group g of row i)
    const int lg = lane & 3, from4 = 4 * (4 * i + q);
#pragma unroll
    for (int t = 0; t < TJ; t++) {
        const int r = n0 + 16 * (glu ? t >> 1 : t) + (lane >> 2);
        row[t] = (glu && (t & 1) ? w2 : w) + (size_t)(r < n ? r : n - 1) * row_bytes;
    }
    // x: octet lane & 15 of the unit, vectors lane >> 4 and, with eight vectors, 4 + (lane >> 4)
    const float *xl[P];
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int v = 4 * p + q;
        xl[p] = x + (size_t)(v < m ? v : m - 1) * k + 8 * i;
    }
    uint8_t *const area = lds + wave * x_bytes<MV>();
    float *const area_inv = reinterpret_cast<float *>(area + 2 * MV * XROW);
    uint8_t *xw[P];
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int o = i & 3;                                      // octet of group i >> 2
        const int at = WF::ORDER <= OCTET_SWAPPED ? row_part(WF::ORDER, o) * 16 : (o >> 1) * 8;
        xw[p] = area + (4 * p + q) * XROW + (i >> 2) * 64 + at;
    }
    // (halves: an octet is two operand halves, of the lane rows of parts 2 (o & 1) and 2 (o & 1) + 1)
    const int h0 = WF::ORDER > OCTET_SWAPPED ? row_part(WF::ORDER, 2 * (i & 1)) * 16 : 0;
    const int h1 = WF::ORDER > OCTET_SWAPPED ? row_part(WF::ORDER, 2 * (i & 1) + 1) * 16 : 0;
    const uint8_t *const xrd = area + (i & (2 * MV - 1)) * XROW + q * 16;

    WF raw[D][TJ];
    v4f xr[P][2], nr[2];
    auto load_w = [&](WF (&dst)[TJ], int u) __attribute__((always_inline)) {
        const int uc = u < units ? u : units - 1;
        const int g = 4 * uc + lg < groups ? lg : groups - 1 - 4 * uc;  // (past the row's end: its last group, with scale 0)
#pragma unroll
        for (int t = 0; t < TJ; t++) dst[t].load(row[t], uc, g);
    };
    auto load_x = [&](int u) __attribute__((always_inline)) {
        const int uc = u < units ? u : units - 1;
        const int at = 128 * uc + 8 * i < k ? 128 * uc : 128 * uc - 32 * (i >> 2);   // (past the end: the unit's first group)
#pragma unroll
        for (int p = 0; p < P; p++) {
            xr[p][0] = *reinterpret_cast<const v4f_a4 *>(xl[p] + at);
            xr[p][1] = *reinterpret_cast<const v4f_a4 *>(xl[p] + at + 4);
        }
        if constexpr (NORM) {
            nr[0] = *reinterpret_cast<const v4f *>(norm_w + 8 * i + at);
            nr[1] = *reinterpret_cast<const v4f *>(norm_w + 8 * i + at + 4);
        }
    };
    float ss[P];                                                  // NORM: this lane's part of its vectors' sums of squares
#pragma unroll
    for (int p = 0; p < P; p++) ss[p] = 0.0f;
    // This lane's octets of unit u, and the biased exponent of the vector's largest |x| in the unit.
    float e[P][8];
    int ex[P];
    auto take_x = [&](int u) __attribute__((always_inline)) {
        const bool past = 128 * u + 8 * i >= k;
#pragma unroll
        for (int p = 0; p < P; p++) {
#pragma unroll
            for (int c = 0; c < 8; c++) {
                if constexpr (MOVED) asm("v_mov_b32 %0, %1" : "=&v"(e[p][c]) : "v"(xr[p][c >> 2][c & 3]));
                else e[p][c] = xr[p][c >> 2][c & 3];
            }
            if (Fmt<FMT>::BE < 128 && past) {
#pragma unroll
                for (int c = 0; c < 8; c++) e[p][c] = 0.0f;
            }
            if constexpr (NORM) {
                if (u < units) {
#pragma unroll
                    for (int c = 0; c < 8; c++) ss[p] = __builtin_fmaf(e[p][c], e[p][c], ss[p]);
                }
#pragma unroll
                for (int c = 0; c < 8; c++) e[p][c] *= nr[c >> 2][c & 3];
            }
            const float mx = max3_abs(max3_abs(e[p][0], e[p][1], e[p][2]), max3_abs(e[p][3], e[p][4], e[p][5]), max3_abs(e[p][6], e[p][7], 0.0f));
            ex[p] = (int)(max16(__float_as_uint(mx)) >> 23);
        }
    };
    double acc[TJ][4];
#pragma unroll
    for (int t = 0; t < TJ; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[t][r] = 0.0;
    const v4u ones = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};

    // READY: a unit's operands and inverse scales, fetched with its weights
    v4u xq[D][4];
    v4f iq[D];
    const int xi = i & (2 * MV - 1), xv = xi & (MV - 1);
    const float *const iq_lane = READY ? reinterpret_cast<const float *>(ready + (size_t)units * (512 * m)) + (4 * q & (MV - 1)) : nullptr;
    const uint8_t *const xq_lane = READY ? ready + (q * (2 * m) + (xv < m ? xv : m - 1) + (xi < MV ? 0 : m)) * 16 : nullptr;
    auto load_ready = [&](int d, int u) __attribute__((always_inline)) {
        const int uc = u < units ? u : units - 1;
#pragma unroll
        for (int j = 0; j < 4; j++) xq[d][j] = *reinterpret_cast<const v4u *>(xq_lane + (size_t)uc * (512 * m) + j * (128 * m));
        iq[d] = *reinterpret_cast<const v4f *>(iq_lane + (size_t)uc * 8);
    };
    if constexpr (!READY) load_x(wave);
#pragma unroll
    for (int d = 0; d < D; d++) {
        load_w(raw[d], wave + d * waves);
        if constexpr (READY) load_ready(d, wave + d * waves);
    }
    if constexpr (AHEAD) {
        take_x(wave);
        load_x(wave + waves);
    }

    for (int u0 = wave; u0 < units; u0 += D * waves) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int u = u0 + d * waves;
            if (u < units) {
                if constexpr (!AHEAD && !READY) {
                    take_x(u);
                    load_x(u + waves);
                }
                // (a sum of 32 codes times 2^15 is below 2^28: a block scale from 2^100 on could take it past the largest
                // float where the result, with small x, is not)
                bool large = false;
                if constexpr (F32_SCALE) {
#pragma unroll
                    for (int t = 0; t < TJ; t++) large |= fabsf(__uint_as_float(raw[d][t].r[0])) >= 0x1p100f;
                    large = __builtin_amdgcn_ballot_w64(large) != 0;
                }
                if constexpr (!READY) {
                    // (with such a scale x loses bits below 2^-11 of the largest)
                    int top = 14;
                    if constexpr (F32_SCALE)
                        if (large) top = -14;
                    wave_order();                                 // (the unit before has been read)
                    float s[P], inv_s[P];
                    unsigned long long infinite = 0;
#pragma unroll
                    for (int p = 0; p < P; p++) {
                        if (INFINITIES && keep_infinities) infinite |= __builtin_amdgcn_ballot_w64(ex[p] == 255);
                        octet_scale<F32_SCALE>(ex[p], top, s[p], inv_s[p]);
                        if (i == 0) area_inv[4 * p + q] = inv_s[p];
                    }
#pragma unroll
                    for (int p = 0; p < P; p++) {
                        uint32_t hi[4], lo[4];
                        split_octet<WF::PAIRS>(e[p], s[p], inv_s[p], hi, lo);
                        if constexpr (WF::ORDER <= OCTET_SWAPPED) {
                            *reinterpret_cast<v4u *>(xw[p]) = v4u{hi[0], hi[1], hi[2], hi[3]};
                            *reinterpret_cast<v4u *>(xw[p] + MV * XROW) = v4u{lo[0], lo[1], lo[2], lo[3]};
                        } else {
                            *reinterpret_cast<v2u *>(xw[p] + h0) = v2u{hi[0], hi[1]};
                            *reinterpret_cast<v2u *>(xw[p] + h1) = v2u{hi[2], hi[3]};
                            *reinterpret_cast<v2u *>(xw[p] + MV * XROW + h0) = v2u{lo[0], lo[1]};
                            *reinterpret_cast<v2u *>(xw[p] + MV * XROW + h1) = v2u{lo[2], lo[3]};
                        }
                    }
                    if constexpr (INFINITIES) {
                        // (in LDS, where this costs the usual path no registers)
                        if (__builtin_expect(infinite != 0, 0)) {
#pragma unroll
                            for (int p = 0; p < P; p++)
#pragma unroll
                                for (int c = 0; c < 2; c++) {
                                    uint8_t *const at = xw[p] + (WF::ORDER <= OCTET_SWAPPED ? 8 * c : c ? h1 : h0);
                                    const v2u h = *reinterpret_cast<const v2u *>(at);
                                    v2u l = *reinterpret_cast<const v2u *>(at + MV * XROW);
#pragma unroll
                                    for (int r = 0; r < 2; r++) l[r] = without_infinities(h[r], l[r]);
                                    *reinterpret_cast<v2u *>(at + MV * XROW) = l;
                                }
                        }
                    }
                }
                WF cur[TJ];
#pragma unroll
                for (int t = 0; t < TJ; t++) {
                    cur[t] = placed<FMT>(raw[d][t], from4);
                    cur[t].open(u, Fmt<FMT>::BE < 128 && 4 * u + q >= groups);
                }
                if constexpr (READY && F32_SCALE) {
                    if (__builtin_expect(large, 0)) {
#pragma unroll
                        for (int t = 0; t < TJ; t++)
#pragma unroll
                            for (int j = 0; j < 4; j++) cur[t].sc4[j] *= 0x1p-28f;
                    }
                }
                if constexpr (!READY) wave_order();
                float sum[TJ][4];                                 // of this unit, in units of the vectors' inverse scales
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v4u xa;
                    if constexpr (READY) xa = xq[d][j];
                    else xa = *reinterpret_cast<const v4u *>(xrd + j * 64);
                    v4f xs[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                    if constexpr (WF::MINS) contract<false>(xa, ones, xs);
#pragma unroll
                    for (int t = 0; t < TJ; t++) {
                        const v4u wf = cur[t].frag(j);
                        v4f p[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                        contract<WF::SPLIT16>(xa, wf, p);
                        const float s0 = cur[t].sc(j, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) sum[t][r] = j == 0 ? s0 * p[0][r] : __builtin_fmaf(s0, p[0][r], sum[t][r]);
                        if constexpr (WF::SPLIT16) {
                            const float s1 = cur[t].sc(j, 1);
#pragma unroll
                            for (int r = 0; r < 4; r++) sum[t][r] = __builtin_fmaf(s1, p[1][r], sum[t][r]);
                        }
                        if constexpr (WF::MINS) {
                            const float mn = cur[t].mn(j);
#pragma unroll
                            for (int r = 0; r < 4; r++) sum[t][r] = __builtin_fmaf(mn, xs[0][r], sum[t][r]);
                        }
                    }
                }
                v4f inv;
                if constexpr (READY) inv = iq[d];
                else inv = *reinterpret_cast<const v4f *>(area_inv + (4 * q & (MV - 1)));
                const double back = READY && F32_SCALE && large ? 0x1p28 : 1.0;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    double iv = (double)inv[r];
                    if constexpr (READY && F32_SCALE) iv *= back;
#pragma unroll
                    for (int t = 0; t < TJ; t++) acc[t][r] = __builtin_fma((double)sum[t][r], iv, acc[t][r]);
                }
                if constexpr (AHEAD) {
                    take_x(u + waves);
                    load_x(u + 2 * waves);
                }
            }
            load_w(raw[d], u + D * waves);
            if constexpr (READY) load_ready(d, u + D * waves);
        }
    }
    // red[wave][vector][16 * TJ rows]; lane rows 0 .. P - 1 hold the hi parts of vectors 0 .. MV - 1, the next P the lo parts
    __syncthreads();
    float *const red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < TJ; t++) {
            const double lo = __shfl_xor(acc[t][r], 16 * P);
            if (q < P) red[(wave * MV + 4 * q + r) * (16 * TJ) + 16 * t + i] = (float)__builtin_fma(lo, 0x1p-11, acc[t][r]);
        }
    float *const squares = red + waves * MV * (16 * TJ);
    if constexpr (NORM && READY) {
        // (a vector's units over the lanes of a wavefront)
        for (int v = wave; v < m; v += waves) {
            const float *const sq = reinterpret_cast<const float *>(ready + ready_squares(m, units));
            double sum = 0.0;
            for (int u = lane; u < units; u += 64) sum += (double)sq[u * 8 + v];
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o);
            if (lane == 0) reinterpret_cast<double *>(squares)[v] = sum;
        }
    } else if constexpr (NORM) {
#pragma unroll
        for (int p = 0; p < P; p++) {
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) ss[p] += __shfl_xor(ss[p], o);
            if (i == 0) squares[wave * MV + 4 * p + q] = ss[p];
        }
    }
    __syncthreads();
    auto total = [&](int v, int c) __attribute__((always_inline)) {
        double sum = 0.0;
        for (int wv = 0; wv < waves; wv++) sum += (double)red[(wv * MV + v) * (16 * TJ) + c];
        return sum;
    };
    const int cols = glu ? 8 * TJ : 16 * TJ;
    for (int o = tid; o < MV * cols; o += (int)blockDim.x) {
        const int v = o / cols, c = o % cols;
        if (v >= m || n0 + c >= n) continue;
        double rinv = 1.0;
        if constexpr (NORM) {                                     // (one step of Newton's iteration: an error here is the whole vector's)
            double sq = 0.0;
            if constexpr (READY) sq = reinterpret_cast<const double *>(squares)[v];
            else for (int wv = 0; wv < waves; wv++) sq += (double)squares[wv * MV + v];
            if (!(sq <= 3.40282347e+38)) {                        // (rarely: as the norm alone has it, x / infinity)
                float zero = 0.0f;                                // (NaN with an infinity or a NaN in x; no early end, so that loads run ahead)
#pragma unroll 4
                for (int j = 0; j < k; j += 4) {
                    const v4f o = *reinterpret_cast<const v4f_a4 *>(x + (size_t)v * k + j);
#pragma unroll
                    for (int e4 = 0; e4 < 4; e4++) zero = __builtin_fmaf(o[e4], 0.0f, zero);
                }
                y[(size_t)v * n + n0 + c] = fabsf(zero);
                continue;
            }
            const double mean = __builtin_fma(sq, 1.0 / (double)k, (double)eps), r0 = (double)(1.0f / sqrtf((float)mean));
            rinv = r0 <= 3.40282347e+38 ? r0 * __builtin_fma(-0.5 * mean, r0 * r0, 1.5) : r0;
        }
        if (glu) {
            const int at = 32 * (c >> 4) + (c & 15);
            const float gate = (float)(total(v, at) * rinv), up = (float)(total(v, at + 16) * rinv);
            y[(size_t)v * n + n0 + c] = gate * (up * (1.0f / (1.0f + expf(-up))));
        } else {
            y[(size_t)v * n + n0 + c] = (float)(total(v, c) * rinv);
        }
    }
}

// ---- float16 a, m <= 16 * MT -----------------------------------------------------------------------------------------
// Rows [m, k] go global -> registers (four lanes per row and group, 64 consecutive bytes) -> the wavefront's part of LDS ->
// operands.  Arranged activations (ARR, the order arrange_a_kernel writes: unit (32 rows, 64 k) of 4 KiB, octet c of half h
// of row fr at ((c * 64) + 32 h + fr) * 16 bytes, its dwords the element pairs (0,4)(1,5)(2,6)(3,7)) are loaded as operands
// where a lane takes whole octets, through LDS where it takes halves of two.
// TURN: activations are brought into the order of the codes after all.
template <int ORDER, int PAIRS, bool ARR, bool TURN = false> struct A16 {
    static constexpr bool OCT = ORDER <= OCTET_SWAPPED;
    static constexpr bool STAGED = !ARR || !OCT;
    static_assert(!TURN || (ARR ? OCT && PAIRS == P01 : PAIRS == P02), "orders that a turn is written for");
    v4u v;
    __device__ __forceinline__ void load(const uint8_t *p, uint32_t at) { v = *reinterpret_cast<const v4u *>(p + at); }
    // the order in which the operand holds an octet: as it comes, but in order where halves of it go to different lanes
    static constexpr int AS = TURN ? PAIRS : ARR && OCT ? (int)P04 : (int)P01;
    __device__ __forceinline__ v4u ordered() const
    {
        constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;
        if constexpr (ARR && (TURN || !OCT))
            return v4u{__builtin_amdgcn_perm(v[1], v[0], LO), __builtin_amdgcn_perm(v[3], v[2], LO),
                       __builtin_amdgcn_perm(v[1], v[0], HI), __builtin_amdgcn_perm(v[3], v[2], HI)};
        else if constexpr (TURN)
            return v4u{__builtin_amdgcn_perm(v[1], v[0], LO), __builtin_amdgcn_perm(v[1], v[0], HI),
                       __builtin_amdgcn_perm(v[3], v[2], LO), __builtin_amdgcn_perm(v[3], v[2], HI)};
        else return v;
    }
};

// A 16-row, 32-k operand in LDS: where row `row` of lane row `part` lies.  One group: lane rows 64 bytes askew.  A pair of groups: the
// rows are turned by four places per lane row and two for the second group, so that the sixteen lanes that write beside
// each other (the 128 bytes of two rows) meet sixteen different places, as the sixteen that read do.
template <bool PAIR> constexpr int ABLK = PAIR ? 1024 : 4 * (256 + 64);
template <bool PAIR> __device__ __forceinline__ int a_place(int part, int row, int group)
{
    return PAIR ? part * 256 + ((row + 4 * part + 2 * group) & 15) * 16 : part * 320 + row * 16;
}
// Rows of a are fetched as pairs of groups, by which eight operands beside two row tiles would spill: those take single groups.  So do
// the forms for two workgroups to a CU that spilled in pairs and lost by it (GGUF_Q4_0 200 x 1280 -> 5120 15.2 / 16.9 us, Q4_K 37 x
// 2048 -> 9000 15.9 / 16.6, Q6_K 64 x 4096 -> 14336 30.9 / 32.3).
constexpr bool in_pairs(int fmt, int mt, bool arr, bool full)
{
    const bool spills = mt == 4 ? fmt == RFQ_Q4_0 || fmt == RFQ_GGUF_Q4_0 || fmt == RFQ_Q6_K : mt == 3 && fmt == RFQ_Q4_K;
    return !arr && mt < 8 && !(full && spills);
}
template <int MT, int TJ, bool STAGED, bool PAIR> constexpr int gemm_lds(int waves)
{
    constexpr int A = STAGED ? (PAIR ? 2 : 1) * MT * ABLK<PAIR> : 0, RED = 16 * MT * 16 * TJ * 4;
    return waves * (A > RED ? A : RED);
}

// blockDim = 64 * waves; LDS: gemm_lds.  a: rows [m, k] or the arranged buffer; blockIdx.y: slices of rows_per_slice (a
// multiple of 16, at most 16 * MT) rows each.
// FULL: for more workgroups than CUs, two of them to a CU (128 registers).  PAIR: rows are fetched as pairs of groups; DEEP: two
// pairs ahead.  TURN: see A16.
template <int FMT, int MT, int TJ, bool ARR, int D, int WAVES, bool FULL, bool PAIR, bool DEEP, bool TURN>
__global__ void __launch_bounds__(64 * WAVES, FULL && (PAIR || ARR) ? 4 : 1)
gemm_skinny_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ a, void *__restrict__ y, int f16_out, int m, int n, int k,
                   int rows_per_slice)
{
    typedef W<FMT> WF;
    typedef A16<WF::ORDER, WF::PAIRS, ARR, TURN> AF;
    constexpr int PAIRS_AHEAD = DEEP ? 2 : 1;
    constexpr int AD = PAIR ? 2 * PAIRS_AHEAD : MT <= 2 ? 4 : MT * TJ < 12 ? 2 : 1;  // groups of activations in flight (registers)
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int groups = k >> 5, units = groups >> 2;               // (whole units; what is left of a row comes after them)
    const int n0 = blockIdx.x * (16 * TJ);
    const size_t row_bytes = (size_t)(k / Fmt<FMT>::BE) * Fmt<FMT>::BB;
    const uint8_t *row[TJ];                                       // (weights: lane 4 * i + g fetches group g of row i)
    const int lg = lane & 3, from4 = 4 * (4 * i + q);
#pragma unroll
    for (int t = 0; t < TJ; t++) {
        const int r = n0 + 16 * t + (lane >> 2);
        row[t] = w + (size_t)(r < n ? r : n - 1) * row_bytes;
    }
    const int m0 = blockIdx.y * rows_per_slice;
    // Arranged: a lane takes its row's octet.  Rows: eight lanes take the 128 bytes of two neighbouring groups of a row, whole cache
    // lines (with the 64 bytes of one group every line came twice from L2, which bound the kernel: Q8_0, 96 rows, 4096 ->
    // 4096 3.56 million requests, 20.7 -> 15.8 us).
    const uint8_t *al[PAIR ? 1 : MT];
    uint32_t ao[PAIR ? MT : 1][2];
    const uint8_t *const a0 = PAIR ? a + (size_t)m0 * k * 2 : nullptr;
    if constexpr (!PAIR) {
        const size_t nst = (size_t)((k + 63) / 64);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            int r = m0 + 16 * t + (ARR ? i : lane >> 2);
            r = r < m ? r : m - 1;
            if constexpr (ARR) al[t] = a + (size_t)(r >> 5) * nst * 4096 + (r & 31) * 16 + (AF::OCT ? row_part(WF::ORDER, q) : q) * 1024;
            else al[t] = a + ((size_t)r * k + 8 * lg) * 2;
        }
    } else {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int r = 16 * t + 8 * e + (lane >> 3), last = m - m0 - 1;
                ao[t][e] = (uint32_t)(r < last ? r : last) * (uint32_t)(2 * k) + 16 * (lane & 7);
            }
    }
    // staging: the lane that holds octet `oct` of row `r16` (of the pair's group `gs`) writes where lane row row_part(octet) reads
    // (halves: two pieces)
    constexpr int BLK = ABLK<PAIR>, PLANE = MT * BLK;
    uint8_t *const area = lds + wave * ((PAIR ? 2 : 1) * PLANE);
    const int r16 = ARR ? i : PAIR ? lane >> 3 : lane >> 2, oct = ARR ? q : lane & 3, gs = PAIR ? (lane >> 2) & 1 : 0;
    const int st0 = gs * PLANE + (AF::OCT ? a_place<PAIR>(row_part(WF::ORDER, oct), r16, gs) : a_place<PAIR>(2 * (oct & 1), r16, gs) + 8 * (oct >> 1));
    const int st1 = AF::OCT ? 0 : gs * PLANE + a_place<PAIR>(2 * (oct & 1) + 1, r16, gs) + 8 * (oct >> 1);
    const int rd[2] = {a_place<PAIR>(q, i, 0), PAIR ? PLANE + a_place<PAIR>(q, i, 1) : 0};

    WF raw[D][TJ];
    AF ar[AD][MT];
    auto load_w = [&](WF (&dst)[TJ], int u) __attribute__((always_inline)) {
        const int uc = u < units ? u : units > 0 ? units - 1 : 0;
        const int g = 4 * uc + lg < groups ? lg : groups - 1 - 4 * uc;  // (past the row's end: its last group)
#pragma unroll
        for (int t = 0; t < TJ; t++) dst[t].load(row[t], uc, g);
    };
    auto load_a = [&](AF (&dst)[MT], int u, int j) __attribute__((always_inline)) {
        if constexpr (!PAIR) {
            int g = 4 * u + j;
            g = g < groups ? g : groups - 1;
            const uint32_t at = ARR ? (uint32_t)(g >> 1) * 4096u + (g & 1) * 512u : (uint32_t)g * 64u;
#pragma unroll
            for (int t = 0; t < MT; t++) dst[t].load(al[t], at);
        }
    };
    // groups 2 p and 2 p + 1 of unit u: rows 8 e .. 8 e + 7 of each operand into ar[2 slot + e] (back: bytes to step back where the second
    // group lies past the end of the row)
    auto load_pair = [&](int slot, int u, int p, uint32_t back) __attribute__((always_inline)) {
        if constexpr (PAIR) {
            const uint8_t *const at = a0 + (size_t)(2 * u + p) * 128;
#pragma unroll
            for (int t = 0; t < MT; t++)
#pragma unroll
                for (int e = 0; e < 2; e++) ar[2 * slot + e][t].load(at, ao[t][e] - back);
        }
    };
    float acc[MT][TJ][4];
#pragma unroll
    for (int b = 0; b < MT; b++)
#pragma unroll
        for (int t = 0; t < TJ; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[b][t][r] = 0.0f;
    const v4u ones = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};

    if constexpr (!PAIR) {
#pragma unroll
        for (int j = 0; j < AD; j++) load_a(ar[j], wave, j);
    } else if (units > 0) {
#pragma unroll
        for (int p = 0; p < PAIRS_AHEAD; p++) load_pair(p, wave < units ? wave : units - 1, p, 0);
    }
#pragma unroll
    for (int d = 0; d < D; d++) load_w(raw[d], wave + d * waves);

    auto put = [&](const AF &src, int b, int turn) __attribute__((always_inline)) {
        const v4u o = src.ordered();
        if constexpr (AF::OCT) {
            *reinterpret_cast<v4u *>(area + b * BLK + (st0 ^ turn)) = o;
        } else {
            *reinterpret_cast<v2u *>(area + b * BLK + (st0 ^ turn)) = v2u{o[0], o[1]};
            *reinterpret_cast<v2u *>(area + b * BLK + (st1 ^ turn)) = v2u{o[2], o[3]};
        }
    };
    // a pair of groups to LDS (rows 8 .. 15: eight places further round)
    auto put_pair = [&](int slot) __attribute__((always_inline)) {
        if constexpr (PAIR) {
            wave_order();                                         // (the pair before has been read)
#pragma unroll
            for (int b = 0; b < MT; b++) { put(ar[2 * slot][b], b, 0); put(ar[2 * slot + 1][b], b, 128); }
            wave_order();
        }
    };
    auto get = [&](int g, v4u (&xa)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < MT; b++) xa[b] = *reinterpret_cast<const v4u *>(area + b * BLK + rd[g]);
    };
    // one group's activations to operands
    auto operands = [&](const AF (&src)[MT], v4u (&xa)[MT]) __attribute__((always_inline)) {
        if constexpr (!AF::STAGED) {
#pragma unroll
            for (int b = 0; b < MT; b++) xa[b] = src[b].ordered();
        } else {
            wave_order();                                         // (the group before has been read)
#pragma unroll
            for (int b = 0; b < MT; b++) put(src[b], b, 0);
            wave_order();
            get(0, xa);
        }
    };
    auto multiply = [&](const WF (&cur)[TJ], const v4u (&xa)[MT], int j) __attribute__((always_inline)) {
        v4u wf[TJ];
        float s0[TJ], s1[TJ], mn[TJ];
#pragma unroll
        for (int t = 0; t < TJ; t++) {
            wf[t] = cur[t].template frag_as<AF::AS>(j);
            s0[t] = cur[t].sc(j, 0);
            s1[t] = WF::SPLIT16 ? cur[t].sc(j, 1) : 0.f;
            mn[t] = WF::MINS ? cur[t].mn(j) : 0.f;
        }
#pragma unroll
        for (int b = 0; b < MT; b++) {
            v4f xs[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            if constexpr (WF::MINS) contract<false>(xa[b], ones, xs);
#pragma unroll
            for (int t = 0; t < TJ; t++) {
                v4f p[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                contract<WF::SPLIT16>(xa[b], wf[t], p);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    acc[b][t][r] = __builtin_fmaf(s0[t], p[0][r], acc[b][t][r]);
                    if constexpr (WF::SPLIT16) acc[b][t][r] = __builtin_fmaf(s1[t], p[1][r], acc[b][t][r]);
                    if constexpr (WF::MINS) acc[b][t][r] = __builtin_fmaf(mn[t], xs[0][r], acc[b][t][r]);
                }
            }
        }
    };
    for (int u0 = wave; u0 < units; u0 += D * waves) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int u = u0 + d * waves;
            if (u < units) {
                WF cur[TJ];
#pragma unroll
                for (int t = 0; t < TJ; t++) {
                    cur[t] = placed<FMT>(raw[d][t], from4);
                    cur[t].open(u, false);
                    cur[t].template turn<AF::AS>();
                }
                if constexpr (PAIR) {
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        constexpr int P2 = PAIRS_AHEAD == 2;
                        const int next = u + waves < units ? u + waves : units - 1;
                        put_pair(P2 ? p : 0);
                        load_pair(P2 ? p : 0, !P2 && p == 0 ? u : next, P2 ? p : p ^ 1, 0);
#pragma unroll
                        for (int g = 0; g < 2; g++) {
                            v4u xa[MT];
                            get(g, xa);
                            multiply(cur, xa, 2 * p + g);
                            if constexpr (MT >= 6) __builtin_amdgcn_sched_barrier(0);   // (the groups' operands side by side would not fit the registers)
                        }
                    }
                } else
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v4u xa[MT];
                    operands(ar[j % AD], xa);
                    load_a(ar[j % AD], j + AD < 4 ? u : u + waves, (j + AD) % 4);
                    if constexpr (!AF::STAGED) __builtin_amdgcn_sched_barrier(0);   // (the loads go out before the group is multiplied)
                    multiply(cur, xa, j);
                    if constexpr (MT >= 6) __builtin_amdgcn_sched_barrier(0);   // (the groups' operands side by side would not fit the registers)
                }
            }
            load_w(raw[d], u + D * waves);
        }
    }
    if constexpr (Fmt<FMT>::BE < 128) {
        // The one to three groups behind the last whole unit, by the wavefront whose turn it is.  (As a unit filled up with
        // zeros they would turn an infinity into NaN; a test before every group cost short rows 7 %.)
        if ((groups & 3) != 0 && wave == units % waves) {
            WF cur[TJ];
#pragma unroll
            for (int t = 0; t < TJ; t++) {
                WF last;
                last.load(row[t], units, 4 * units + lg < groups ? lg : 0);
                cur[t] = placed<FMT>(last, from4);
                cur[t].open(units, 4 * units + q >= groups);
                cur[t].template turn<AF::AS>();
            }
            if constexpr (!PAIR) {
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    if (4 * units + j < groups) {
                        AF tail[MT];
                        v4u xa[MT];
                        load_a(tail, units, j);
                        operands(tail, xa);
                        multiply(cur, xa, j);
                    }
                }
            } else {
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    if (4 * units + 2 * p >= groups) continue;
                    const bool both = 4 * units + 2 * p + 1 < groups;
                    load_pair(0, units, p, both ? 0u : 16u * (lane & 4));
                    put_pair(0);
#pragma unroll
                    for (int g = 0; g < 2; g++) {
                        if (g == 1 && !both) continue;
                        v4u xa[MT];
                        get(g, xa);
                        multiply(cur, xa, 2 * p + g);
                    }
                }
            }
        }
    }
    // red[wave][row of a][16 * TJ rows of w]
    __syncthreads();
    float *const red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int b = 0; b < MT; b++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < TJ; t++) red[(wave * (16 * MT) + 16 * b + 4 * q + r) * (16 * TJ) + 16 * t + i] = acc[b][t][r];
    __syncthreads();
    for (int o = tid; o < 16 * MT * 16 * TJ; o += (int)blockDim.x) {
        const int v = o / (16 * TJ), c = o % (16 * TJ);
        if (v >= rows_per_slice || m0 + v >= m || n0 + c >= n) continue;
        float sum = 0.0f;
        for (int wv = 0; wv < waves; wv++) sum += red[(wv * (16 * MT) + v) * (16 * TJ) + c];
        const size_t at = (size_t)(m0 + v) * n + n0 + c;
        if (f16_out) reinterpret_cast<_Float16 *>(y)[at] = (_Float16)sum;
        else reinterpret_cast<float *>(y)[at] = sum;
    }
}

} // namespace skinny
} // namespace rfq
