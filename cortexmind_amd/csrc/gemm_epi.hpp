// What the fp32 GEMM kernels (gemm.hip, gemm_direct.hip) share: the
// accumulator type, the XCD renumbering and the epilogue's arithmetic.
#pragma once

#include "cxm_common.hpp"

namespace cxm {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup b runs on
// XCD b % 8).  Renumbering b so that each XCD gets one contiguous eighth of
// the row-major tile order makes the tiles sharing an XCD's L2 share A rows
// (and B columns), instead of every XCD touching every row block.
__device__ __forceinline__ unsigned xcd_remap(unsigned b, unsigned g) {
    if (g % 8 != 0) return b;
    return (b % 8) * (g / 8) + b / 8;
}

// One element through the epilogue's options, applied with selects; `pre` is
// the element's gate, or C's old value for the SGD update.
__device__ __forceinline__ float epi_value(const Epilogue &e, float v, float bias, float pre) {
    const float t = v * e.lr;  // SGD: matrix_t::sub(W, ScalarOp::mul(G, lr)): two roundings
    const float sgd = pre - t;
    float u = e.bias ? v + bias : v;
    u = (e.act == CXM_ACT_RELU && 0.0f > u) ? 0.0f : u;
    u = e.gate ? u * (pre > 0.0f ? 1.0f : 0.0f) : u;
    return e.sgd ? sgd : u;
}

// The direct kernels (gemm_direct.hip): any shape and dword alignment, A B,
// A B^T and A^T B.  `ring`: the ring kernel would take the product.  Returns
// 1 when it is better left to the kernels of gemm.hip.
int gemm_direct(const float *A, const float *B, float *C, size_t M, size_t K, size_t N, int ta, int tb,
                const Epilogue &epi, bool ring, cxm_stream_t st);

}  // namespace cxm
