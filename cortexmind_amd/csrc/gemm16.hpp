// What the 16-bit GEMM kernels (gemm16.hip, gemm16_direct.hip) share: the
// fragment types, the MFMA and the host entry of the direct kernels.
#pragma once

#include "half.hpp"

namespace cxm {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <int DT>
__device__ __forceinline__ f32x16 mfma16(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (DT == CXM_DT_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
}

}  // namespace

// The direct 16-bit kernels (gemm16_direct.hip): any shape, 2-byte alignment,
// A B, A B^T and A^T B.  `ring`: a ring kernel would take the product; `vec`:
// both operands' stored rows allow the staged kernels' 128-bit loads.
// kDeclined (gemm_epi.hpp): left to the kernels of gemm16.hip.
int gemm16_direct(const uint16_t *A, const uint16_t *B, uint16_t *C, size_t M, size_t K, size_t N, bool ta, bool tb,
                  int dtype, bool ring, bool vec, cxm_stream_t st);

}  // namespace cxm
