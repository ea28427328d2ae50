// Integer codes of weights as fp16 operands (exact: 1024 + code is read from its bits, then 1024 comes off again): what the
// few-row kernels and the tiled kernel on integer codes share.
#pragma once
#include "rfq_common.hpp"

namespace rfq {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t add2h(uint32_t bits, float bias)
{
    v2h h;
    __builtin_memcpy(&h, &bits, 4);
    h = h + v2h{(_Float16)bias, (_Float16)bias};
    uint32_t o;
    __builtin_memcpy(&o, &h, 4);
    return o;
}
// the nibbles at bits SHIFT and SHIFT + 16 of a dword as an fp16 pair of nibble + bias (0x6400 | c reads 1024 + c).  One and-or
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

} // namespace rfq
