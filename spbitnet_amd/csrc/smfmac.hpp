// smfmac.hpp -- what the kernels on v_smfmac_i32_16x16x128_i8 share: operand
// types, the decode of spbitnet's packed ternary words into the sparse A
// operand (the layouts are described in gemm.hip), stacked matrices.
#pragma once

#include <cstdint>

#include "common.hpp"

namespace spb {

// Raises a kernel's dynamic-LDS limit to the CU's LDS, once per device
// (gemm.hip); false if the runtime refuses.
bool gemm_allow_lds(const void* fn);

namespace {

// Up to three matrices stacked along the rows (q | k | v, gate | up), with
// equal columns and strides: rows [0, end0) are the first, [end0, end1) the
// second (words at meta + om1 for global row r, i.e. om1 = offset of the
// second matrix - end0 * ms), [end1, rows) the third.  One matrix: end0 =
// end1 = rows.
struct GemmSegs {
    long om1, om2, ov1, ov2;
    int end0, end1;
};

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
constexpr int kRawBufferFlags = 0x00020000;  // gfx9 raw buffer resource word 3
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

template <uint32_t kTable>
__device__ __forceinline__ uint32_t gemm_bitop3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, kTable);
}

// Index word of one meta word (8 groups): nibble g = p0 | p1 << 2.
__device__ __forceinline__ int smfmac_index(uint32_t k) {
    const uint32_t a = k >> 1, c = k << 1;
    const uint32_t t0 = gemm_bitop3<0x20>(a, k, 0x11111111u);  // (a & ~b) & m : ~b0 & b1
    const uint32_t t1 = gemm_bitop3<0x02>(c, k, 0x22222222u);  // ~(a | b) & m : ~(b0 | b1)
    const uint32_t t2 = gemm_bitop3<0xA2>(a, k, 0x44444444u);  // (a | ~b) & m : b3 | ~b2
    const uint32_t t3 = gemm_bitop3<0xA8>(c, k, 0x88888888u);  // (a | b) & m  : b3 | b2
    return static_cast<int>(gemm_bitop3<0xFE>(t0, t1, t2) | t3);
}

// Four compressed-value dwords (16 int8 +-1) from 16 sign bits: bit j -> byte j.
__device__ __forceinline__ v4i smfmac_values(uint32_t s16) {
    v4i a;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t nib = (s16 >> (4 * d)) & 0xFu;
        const uint32_t nb = (nib * 0x00204081u) & 0x01010101u;  // bit i -> byte i (0/1)
        // per 16-bit half: 0/1 bytes * 0xFE + 0x0101 -> 0x01 / 0xFF bytes, no carries
        u16x2 h = __builtin_bit_cast(u16x2, nb);
        h = h * (u16x2){0xFE, 0xFE} + (u16x2){0x0101, 0x0101};
        a[d] = __builtin_bit_cast(int, h);
    }
    return a;
}

bool gemm_aligned(const void* p, uintptr_t a) {
    return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}

}  // namespace
}  // namespace spb
