// What the GEMM kernels share: the accumulator type, the XCD renumbering and
// the fp32 epilogue's arithmetic (gemm.hip, gemm_direct.hip), the plan and
// the split sum of the direct kernels (gemm_direct.hip, gemm16_direct.hip).
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

// The sum of a float4's split partials (components `plane` floats apart) in
// split order, four splits of loads in flight.
__device__ __forceinline__ float4 sum_splits(const float *p, int plane, unsigned splits, size_t stride) {
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    for (unsigned s0 = 0; s0 < splits; s0 += 4) {
        float4 t[4];
#pragma unroll
        for (unsigned u = 0; u < 4; ++u) {
            const float *d = p + static_cast<size_t>(s0 + u < splits ? s0 + u : splits - 1) * stride;
            t[u] = make_float4(ld_dev(d), ld_dev(d + plane), ld_dev(d + 2 * plane), ld_dev(d + 3 * plane));
        }
#pragma unroll
        for (unsigned u = 0; u < 4; ++u)
            if (s0 + u < splits) {
                a.x += t[u].x; a.y += t[u].y; a.z += t[u].z; a.w += t[u].w;
            }
    }
    return a;
}

// What the direct kernels return for a product that they leave to the others
// (no status code).
constexpr int kDeclined = -1000;

// K splits of a product of 128x128 tiles: where the tiles alone cannot fill
// the chip, at most one workgroup per CU (one fills a CU, and one more would
// run as a second round), each split at least 256 of K.
inline size_t gemm_splits(size_t tiles, size_t K, size_t cus) {
    if (tiles >= cus * 3 / 4 || K < 512) return 1;
    const size_t splits = cus / tiles < K / 256 ? cus / tiles : K / 256;
    return splits < 1 ? 1 : splits;
}

// Tiles and K splits of one product of the direct kernels: about `target`
// workgroups, each split at least `depth` steps of `step` k (a block per wave).
struct DirectPlan {
    size_t tiles, tiles_n, splits, kper;
};
inline DirectPlan direct_plan(size_t M, size_t N, size_t K, size_t tm, size_t tn, size_t step, size_t depth,
                              size_t target) {
    DirectPlan p{};
    p.tiles_n = (N + tn - 1) / tn;
    p.tiles = (M + tm - 1) / tm * p.tiles_n;
    p.splits = 1;
    if (p.tiles < target) {
        p.splits = target / p.tiles;
        const size_t most = K / (depth * step);
        if (p.splits > most) p.splits = most;
        if (p.splits < 1) p.splits = 1;
    }
    p.kper = ((K + p.splits - 1) / p.splits + step - 1) / step * step;
    p.splits = (K + p.kper - 1) / p.kper;
    return p;
}

// The direct kernels (gemm_direct.hip): any shape and dword alignment, A B,
// A B^T and A^T B.  `ring`: the ring kernel would take the product.  Returns
// 1 when it is better left to the kernels of gemm.hip.
int gemm_direct(const float *A, const float *B, float *C, size_t M, size_t K, size_t N, int ta, int tb,
                const Epilogue &epi, bool ring, int vecs, cxm_stream_t st);

}  // namespace cxm
