// Matrix-core contraction for few rows of activations:  y[m, n] = x[m, k] . dequant(W)[n, k]^T, one launch, no temporary.
//
// float16 a, prompts up to about 160 rows (rfq_gemm_f16, rfq_gemm_f16_arranged; prefer_skinny_gemm draws the line).
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
//   * No split of k over workgroups: the wavefronts of a workgroup share 16 * TJ weight rows, take the 128-element units
//     of k in turn and add their results through LDS: one launch, nothing to allocate.
// Measured (cold weights, captured launches; the tiled kernel with its arrangement and its parts -> this one):
//   37 x 4096 -> 4096      Q8_0 33.6 -> 10.7 us   GGUF_Q4_K 25.8 -> 10.5   GGUF_Q6_K 43.0 -> 12.3   Q4_K 22.2 -> 12.6
//   9 x 1024 -> 1000       Q8_0 27.5 -> 3.1       GGUF_Q4_K 20.0 -> 3.2    GGUF_Q6_K 36.0 -> 4.3    Q4_K 16.1 -> 3.9
//   48 x 4096 -> 14336     Q8_0 66.5 -> 32.7      GGUF_Q4_K 42.5 -> 23.3   GGUF_Q6_K 77.9 -> 42.0   Q4_K 40.6 -> 34.7
// (10.5 us for 37 rows of GGUF_Q4_K is 0.9 TB/s of weights: what bounds it is the activations, 384 KB per workgroup
// through LDS, and the instructions, about 60 per unit and 16-row operand.)
#pragma once
#include "rfq_common.hpp"

namespace rfq {
namespace skinny {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

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

__device__ __forceinline__ uint32_t add2h(uint32_t bits, float bias)
{
    v2h h;
    __builtin_memcpy(&h, &bits, 4);
    h = h + v2h{(_Float16)bias, (_Float16)bias};
    uint32_t o;
    __builtin_memcpy(&o, &h, 4);
    return o;
}
// nibbles (n, n + 4) of a dword, n = shift / 4, as an fp16 pair of code + bias (0x6400 | c reads 1024 + c).  One and-or
// after the shift: the instruction takes no literal here, so the mask is kept in a scalar and the magic in a vector register.
template <int SHIFT> __device__ __forceinline__ uint32_t nib2h(uint32_t d, float bias)
{
    uint32_t mask = 0x000F000Fu, magic = 0x64006400u;
    asm("" : "+s"(mask));
    asm("" : "+v"(magic));
    return add2h(((d >> SHIFT) & mask) | magic, bias - 1024.0f);
}
// bytes (0, 1) and (2, 3) of a dword as fp16 pairs of byte + bias
__device__ __forceinline__ void bytes2h(uint32_t d, float bias, uint32_t &p01, uint32_t &p23)
{
    p01 = add2h(__builtin_amdgcn_perm(0x64646464u, d, 0x04010400u), bias - 1024.0f);
    p23 = add2h(__builtin_amdgcn_perm(0x64646464u, d, 0x04030402u), bias - 1024.0f);
}

template <int NW> __device__ __forceinline__ void load_dwords(const uint8_t *a, uint32_t (&d)[NW])
{
    typedef uint32_t v4a4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef uint32_t v2a4 __attribute__((ext_vector_type(2), aligned(4)));
    int i = 0;
#pragma unroll
    for (; i + 4 <= NW; i += 4) {
        const v4a4 v = *reinterpret_cast<const v4a4 *>(a + 4 * i);
        d[i] = v[0]; d[i + 1] = v[1]; d[i + 2] = v[2]; d[i + 3] = v[3];
    }
    if (i + 2 <= NW) {
        const v2a4 v = *reinterpret_cast<const v2a4 *>(a + 4 * i);
        d[i] = v[0]; d[i + 1] = v[1];
        i += 2;
    }
    if (i < NW) d[i] = *reinterpret_cast<const uint32_t *>(a + 4 * i);
}
// Which eight elements of a group lane row q holds, and in which order its four operand dwords hold them.
enum { OCTET, OCTET_SWAPPED, HALVES, HALVES_SWAPPED };           // 8q..  |  8q'..  |  4q.. and 16+4q..  |  4q'.. and 16+4q'..   (q' = q with its bits swapped)
enum { P04, P01, P02 };                                          // (0,4)(1,5)(2,6)(3,7) | (0,1)(2,3)(4,5)(6,7) | (0,2)(1,3)(4,6)(5,7)

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
    __device__ __forceinline__ float sc(int j, int) const { return sc4[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};
template <> struct W<RFQ_Q8_0> : W8<RFQ_Q8_0> {};
template <> struct W<RFQ_GGUF_Q8_0> : W8<RFQ_GGUF_Q8_0> {};

template <> struct W<RFQ_Q4_K> {                                 // 256-byte layout: 8 f16 scales, 8 i8 mins, nibbles at 32 + 28 * sb
    static constexpr int ORDER = OCTET, PAIRS = P04, NR = 7;
    static constexpr bool MINS = true, SPLIT16 = false;
    struct U4 { uint32_t v[4]; };
    uint32_t r[NR], q[4];
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 256u;
        const int h = u & 1;
        uint32_t s[2];
        load_dwords<2>(blk + 8 * h, s);
        r[4] = s[0]; r[5] = s[1];
        r[6] = *reinterpret_cast<const uint32_t *>(blk + 16 + 4 * h);
        const U4 v = ld_once<U4>(blk + 32 + 28 * (4 * h + g));
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = v.v[i];
    }
    __device__ __forceinline__ void open(int, bool)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = r[i];
        transpose4(q[0], q[1], q[2], q[3]);
    }
    __device__ __forceinline__ v4u frag(int j) const { return v4u{nib2h<0>(q[j], 0.f), nib2h<4>(q[j], 0.f), nib2h<8>(q[j], 0.f), nib2h<12>(q[j], 0.f)}; }
    __device__ __forceinline__ float sc(int j, int) const { return f16_bits_to_f32((uint16_t)(r[4 + (j >> 1)] >> (16 * (j & 1)))); }
    __device__ __forceinline__ float mn(int j) const { return (float)(int)(int8_t)(r[6] >> (8 * j)); }
};

template <> struct W<RFQ_GGUF_Q4_K> {
    static constexpr int ORDER = OCTET_SWAPPED, PAIRS = P02, NR = 8;
    static constexpr bool MINS = true, SPLIT16 = false;
    uint32_t r[NR], q[4];
    uint32_t scb, mnb; float d, dm;
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 144u;
        uint32_t a[4], b[4];
        load_dwords<4>(blk, a);
        load_dwords<4>(blk + 16 + 64 * (u & 1) + 16 * g, b);
#pragma unroll
        for (int i = 0; i < 4; i++) { r[i] = b[i]; r[4 + i] = a[i]; }
    }
    // lane row (q1 q0) holds bytes 16 q0 .. of the unit's 64-element chunk q1; it keeps bytes 16 q0 + 8 q1 .. +8 of both
    __device__ __forceinline__ void open(int u, bool)
    {
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = r[i];
        swap32(q[0], q[2]);
        swap32(q[1], q[3]);
        if ((u & 1) == 0) {
            scb = r[5] & 0x3F3F3F3Fu;
            mnb = r[6] & 0x3F3F3F3Fu;
        } else {
            scb = (r[7] & 0x0F0F0F0Fu) | ((r[5] >> 2) & 0x30303030u);
            mnb = ((r[7] >> 4) & 0x0F0F0F0Fu) | ((r[6] >> 2) & 0x30303030u);
        }
        d = f16_bits_to_f32((uint16_t)r[4]);
        dm = -f16_bits_to_f32((uint16_t)(r[4] >> 16));
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        const uint32_t a = q[2 * (j >> 1)], b = q[2 * (j >> 1) + 1];
        if (j & 1) return v4u{nib2h<4>(a, 0.f), nib2h<12>(a, 0.f), nib2h<4>(b, 0.f), nib2h<12>(b, 0.f)};
        return v4u{nib2h<0>(a, 0.f), nib2h<8>(a, 0.f), nib2h<0>(b, 0.f), nib2h<8>(b, 0.f)};
    }
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
        r[6] = *reinterpret_cast<const uint32_t *>(blk + 4 * c);
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
    __device__ __forceinline__ float sc(int j, int h) const { return h ? sb[j] : sa[j]; }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};

template <> struct W<RFQ_GGUF_Q6_K> {
    static constexpr int ORDER = HALVES_SWAPPED, PAIRS = P01, NR = 13;
    static constexpr bool MINS = false, SPLIT16 = true;
    uint32_t r[NR];
    uint32_t a[2], b[2], c[2], s[2]; float d;
    // Eight bytes at p, of which o (0 or 2) lie in the dword before: three aligned dwords, or two and the second again
    static __device__ __forceinline__ void piece(const uint8_t *p, uint32_t o, uint32_t *out)
    {
        uint32_t v[2];
        load_dwords<2>(p - o, v);
        out[0] = v[0]; out[1] = v[1];
        out[2] = *reinterpret_cast<const uint32_t *>(p - o + (o ? 8 : 4));
    }
    __device__ __forceinline__ void load(const uint8_t *row, int u, int g)
    {
        const uint8_t *blk = row + (uint32_t)(u >> 1) * 210u;
        const int half = u & 1;
        const uint32_t o = (uint32_t)(reinterpret_cast<uintptr_t>(blk) & 3u);
        piece(blk + 64 * half + 8 * g, o, r);
        piece(blk + 64 * half + 32 + 8 * g, o, r + 3);
        piece(blk + 128 + 32 * half + 8 * g, o, r + 6);
        piece(blk + 192 + 8 * half, o, r + 9);
        r[12] = *reinterpret_cast<const uint16_t *>(blk + 208) | (o << 16);
    }
    // lane row (q1 q0) holds codes 8 q .. 8 q + 7 (of 32) of every group; after the exchange dword 0 holds four codes of
    // the first 16, dword 1 of the second, both number 2 q0 + q1 of their four
    __device__ __forceinline__ void open(int, bool)
    {
        const uint32_t sel = 0x03020100u + __builtin_amdgcn_perm(0u, r[12] >> 16, 0u);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            a[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel);
            b[i] = __builtin_amdgcn_perm(r[i + 4], r[i + 3], sel);
            c[i] = __builtin_amdgcn_perm(r[i + 7], r[i + 6], sel);
            s[i] = __builtin_amdgcn_perm(r[i + 10], r[i + 9], sel);
        }
        swap32(a[0], a[1]);
        swap32(b[0], b[1]);
        swap32(c[0], c[1]);
        d = f16_bits_to_f32((uint16_t)r[12]);
    }
    __device__ __forceinline__ v4u frag(int j) const
    {
        v4u o;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const uint32_t l = (((j & 1) ? b[e] : a[e]) >> (4 * (j >> 1))) & 0x0F0F0F0Fu;
            const uint32_t t = (j < 2 ? c[e] << (4 - 2 * j) : c[e] >> (2 * j - 4)) & 0x30303030u;
            uint32_t p, r2;
            bytes2h(l | t, -32.f, p, r2);
            o[2 * e] = p;
            o[2 * e + 1] = r2;
        }
        return o;
    }
    __device__ __forceinline__ float sc(int j, int hf) const { const int at = 2 * j + hf; return d * (float)(int)(int8_t)(s[at >> 2] >> (8 * (at & 3))); }
    __device__ __forceinline__ float mn(int) const { return 0.f; }
};

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
    return (order == OCTET_SWAPPED || order == HALVES_SWAPPED) ? ((q & 1) << 1) | (q >> 1) : q;
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

// ---- float16 a, m <= 16 * MT -----------------------------------------------------------------------------------------
// Rows [m, k] go global -> registers (four lanes per row and group, 64 consecutive bytes) -> the wavefront's part of LDS ->
// operands.  Arranged activations (ARR, the order arrange_a_kernel writes: unit (32 rows, 64 k) of 4 KiB, octet c of half h
// of row fr at ((c * 64) + 32 h + fr) * 16 bytes, its dwords the element pairs (0,4)(1,5)(2,6)(3,7)) are loaded as operands
// where a lane takes whole octets, through LDS where it takes halves of two.
template <int ORDER, int PAIRS, bool ARR> struct A16 {
    static constexpr bool OCT = ORDER <= OCTET_SWAPPED;
    static constexpr bool STAGED = !ARR || !OCT;
    v4u v;
    __device__ __forceinline__ void load(const uint8_t *p, uint32_t at) { v = *reinterpret_cast<const v4u *>(p + at); }
    // an octet in operand order
    __device__ __forceinline__ v4u ordered() const
    {
        constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;
        if constexpr (ARR) {
            if constexpr (PAIRS == P04) return v;
            else if constexpr (PAIRS == P01)
                return v4u{__builtin_amdgcn_perm(v[1], v[0], LO), __builtin_amdgcn_perm(v[3], v[2], LO),
                           __builtin_amdgcn_perm(v[1], v[0], HI), __builtin_amdgcn_perm(v[3], v[2], HI)};
            else
                return v4u{__builtin_amdgcn_perm(v[2], v[0], LO), __builtin_amdgcn_perm(v[3], v[1], LO),
                           __builtin_amdgcn_perm(v[2], v[0], HI), __builtin_amdgcn_perm(v[3], v[1], HI)};
        } else if constexpr (PAIRS == P01) return v;
        else if constexpr (PAIRS == P04)
            return v4u{__builtin_amdgcn_perm(v[2], v[0], LO), __builtin_amdgcn_perm(v[2], v[0], HI),
                       __builtin_amdgcn_perm(v[3], v[1], LO), __builtin_amdgcn_perm(v[3], v[1], HI)};
        else
            return v4u{__builtin_amdgcn_perm(v[1], v[0], LO), __builtin_amdgcn_perm(v[1], v[0], HI),
                       __builtin_amdgcn_perm(v[3], v[2], LO), __builtin_amdgcn_perm(v[3], v[2], HI)};
    }
};

constexpr int ABLK = 4 * (256 + 64);                              // bytes of a 16-row, 32-k operand in LDS, lane rows bank-skewed
template <int MT, int TJ, bool STAGED> constexpr int gemm_lds(int waves)
{
    return waves * (STAGED && MT * ABLK > 16 * MT * 16 * TJ * 4 ? MT * ABLK : 16 * MT * 16 * TJ * 4);
}

// blockDim = 64 * waves; LDS: gemm_lds.  a: rows [m, k] or the arranged buffer; blockIdx.y: slices of rows_per_slice (a
// multiple of 16, at most 16 * MT) rows each.
template <int FMT, int MT, int TJ, bool ARR, int D, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
gemm_skinny_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ a, void *__restrict__ y, int f16_out, int m, int n, int k,
                   int rows_per_slice)
{
    typedef W<FMT> WF;
    typedef A16<WF::ORDER, WF::PAIRS, ARR> AF;
    constexpr int AD = MT <= 2 ? 4 : MT * TJ < 12 ? 2 : 1;            // groups of activations in flight (registers)
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int groups = k >> 5, units = (groups + 3) >> 2;
    const int n0 = blockIdx.x * (16 * TJ);
    const size_t row_bytes = (size_t)(k / Fmt<FMT>::BE) * Fmt<FMT>::BB;
    const uint8_t *row[TJ];                                       // (weights: lane 4 * i + g fetches group g of row i)
    const int lg = lane & 3, from4 = 4 * (4 * i + q);
#pragma unroll
    for (int t = 0; t < TJ; t++) {
        const int r = n0 + 16 * t + (lane >> 2);
        row[t] = w + (size_t)(r < n ? r : n - 1) * row_bytes;
    }
    const int part = row_part(WF::ORDER, q), m0 = blockIdx.y * rows_per_slice;
    const uint8_t *al[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) {
        int r = m0 + 16 * t + (ARR ? i : lane >> 2);
        r = r < m ? r : m - 1;
        if constexpr (ARR) {
            const size_t nst = (size_t)((k + 63) / 64);
            al[t] = a + (size_t)(r >> 5) * nst * 4096 + (r & 31) * 16 + (AF::OCT ? part : q) * 1024;
        } else {
            al[t] = a + ((size_t)r * k + 8 * lg) * 2;
        }
    }
    // staging: the lane that holds octet `oct` of row `r16` (rows: lane 4 * row + octet; arranged: 16 * octet + row) writes where lane row row_part(octet) reads (halves: two pieces)
    uint8_t *const area = lds + wave * (MT * ABLK);
    const int r16 = (ARR ? i : lane >> 2) * 16, oct = ARR ? q : lg;
    const int st0 = AF::OCT ? row_part(WF::ORDER, oct) * 320 + r16 : row_part(WF::ORDER, 2 * (oct & 1)) * 320 + r16 + 8 * (oct >> 1);
    const int st1 = AF::OCT ? 0 : row_part(WF::ORDER, 2 * (oct & 1) + 1) * 320 + r16 + 8 * (oct >> 1);
    const int rd = q * 320 + i * 16;

    WF raw[D][TJ];
    AF ar[AD][MT];
    auto load_w = [&](WF (&dst)[TJ], int u) __attribute__((always_inline)) {
        const int uc = u < units ? u : units - 1;
        const int g = 4 * uc + lg < groups ? lg : groups - 1 - 4 * uc;  // (past the row's end: its last group, as zeros)
#pragma unroll
        for (int t = 0; t < TJ; t++) dst[t].load(row[t], uc, g);
    };
    auto load_a = [&](AF (&dst)[MT], int u, int j) __attribute__((always_inline)) {
        int g = 4 * u + j;
        g = g < groups ? g : groups - 1;
        const uint32_t at = ARR ? (uint32_t)(g >> 1) * 4096u + (g & 1) * 512u : (uint32_t)g * 64u;
#pragma unroll
        for (int t = 0; t < MT; t++) dst[t].load(al[t], at);
    };
    float acc[MT][TJ][4];
#pragma unroll
    for (int b = 0; b < MT; b++)
#pragma unroll
        for (int t = 0; t < TJ; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[b][t][r] = 0.0f;
    const v4u ones = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};

#pragma unroll
    for (int j = 0; j < AD; j++) load_a(ar[j], wave, j);
#pragma unroll
    for (int d = 0; d < D; d++) load_w(raw[d], wave + d * waves);

    for (int u0 = wave; u0 < units; u0 += D * waves) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int u = u0 + d * waves;
            if (u < units) {
                WF cur[TJ];
#pragma unroll
                for (int t = 0; t < TJ; t++) {
                    cur[t] = placed<FMT>(raw[d][t], from4);
                    cur[t].open(u, Fmt<FMT>::BE < 128 && 4 * u + q >= groups);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v4u xa[MT];
                    if constexpr (!AF::STAGED) {
#pragma unroll
                        for (int b = 0; b < MT; b++) xa[b] = ar[j % AD][b].ordered();
                    } else {
                        // (a wavefront's LDS operations complete in order: no barrier around its own area)
#pragma unroll
                        for (int b = 0; b < MT; b++) {
                            const v4u o = ar[j % AD][b].ordered();
                            if constexpr (AF::OCT) {
                                *reinterpret_cast<v4u *>(area + b * ABLK + st0) = o;
                            } else {
                                *reinterpret_cast<v2u *>(area + b * ABLK + st0) = v2u{o[0], o[1]};
                                *reinterpret_cast<v2u *>(area + b * ABLK + st1) = v2u{o[2], o[3]};
                            }
                        }
#pragma unroll
                        for (int b = 0; b < MT; b++) xa[b] = *reinterpret_cast<const v4u *>(area + b * ABLK + rd);
                    }
                    load_a(ar[j % AD], j + AD < 4 ? u : u + waves, (j + AD) % 4);
                    v4u wf[TJ];
                    float s0[TJ], s1[TJ], mn[TJ];
                    const bool dead = Fmt<FMT>::BE < 128 && 4 * u + j >= groups;
#pragma unroll
                    for (int t = 0; t < TJ; t++) {
                        wf[t] = cur[t].frag(j);
                        if (Fmt<FMT>::BE < 128) {
#pragma unroll
                            for (int r = 0; r < 4; r++) wf[t][r] = dead ? 0u : wf[t][r];
                        }
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
                    if constexpr (MT >= 6) __builtin_amdgcn_sched_barrier(0);   // (the groups' operands side by side would not fit the registers)
                }
            }
            load_w(raw[d], u + D * waves);
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
