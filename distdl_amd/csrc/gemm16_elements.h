// Pieces shared by the 16-bit MFMA products: element conversions, operand
// descriptions, and the entry of the products that do not fill the chip with
// large tiles.
#ifndef DDL_GEMM16_ELEMENTS_H
#define DDL_GEMM16_ELEMENTS_H
#include "gemm_tiles.h"
#include <hip/hip_fp16.h>

namespace ddl {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

__device__ inline uint16_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if (f != f) return 0x7FC0;
    u += 0x7FFFu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

__device__ inline float bf16_bits_to_f32(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

// 16-bit element <-> fp32, round to nearest even on the way back.
template <bool F16>
__device__ inline float elem_to_f32(uint16_t b) {
    if (F16) {
        __half h;
        __builtin_memcpy(&h, &b, 2);
        return __half2float(h);
    }
    return bf16_bits_to_f32(b);
}
template <bool F16>
__device__ inline uint16_t f32_to_elem(float f) {
    if (F16) {
        const __half h = __float2half_rn(f);
        uint16_t b;
        __builtin_memcpy(&b, &h, 2);
        return b;
    }
    return f32_to_bf16_bits(f);
}

// One operand of the product: element (row, k) at p[row * row_stride + k * k_stride],
// one of the strides being 1.
struct Operand16 {
    const uint16_t* p;
    int64_t row_stride, k_stride;
    bool transposed() const { return row_stride == 1 && k_stride != 1; }
    int64_t ld() const { return transposed() ? k_stride : row_stride; }
};

}  // namespace ddl
#endif  // DDL_GEMM16_ELEMENTS_H
