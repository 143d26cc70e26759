// Elementwise fp32 kernels: same-shape binary ops (pow included), row/column
// broadcast, tensor-op-scalar, unary activations, the fused affine +
// activation forward/backward of the C3 workload, and the SGD update.
//
// Replaces the float4 grid-stride loops of the reference's CUDA path
// (kernels::Binary / kernels::scalar / kernels::Unary,
// source/CortexMind/framework/Engine/Kernels/binary.cuh:15-39,
// scalar.cuh:30-54, unary.cuh:16-40) and the CPU Broadcast::row/col
// (Engine/AVX2/broadcast.cpp:182-388), which has no GPU form there.  The
// aligned forms run as the one-float4-per-thread streaming maps of
// cxm_common.hpp (k_map4, k_zip4, k_rowmap4) with the functors below;
// unaligned pointers take scalar grid-stride loops.
//
// Every op rounds exactly as the reference's scalar expression does: the
// library is built with -ffp-contract=off, so x*s+b is a rounded product
// followed by a rounded sum, never an fma.  ReLU is an explicit select
// (0 > t ? 0 : t), matching _mm256_max_ps(0, t) for -0.0 and NaN.
#include <type_traits>

#include "cxm_common.hpp"
#include "ops.hpp"

namespace cxm {
namespace {

__device__ __forceinline__ float bin(int op, float a, float b) {
    switch (op) {
        case CXM_OP_ADD: return a + b;
        case CXM_OP_SUB: return a - b;
        case CXM_OP_MUL: return a * b;
        case CXM_OP_DIV: return a / b;
        case CXM_OP_MAX: return a > b ? a : b;
        case CXM_OP_MIN: return a < b ? a : b;
        default: return pow_f32(a, b);
    }
}

template <int OP>
__device__ __forceinline__ float4 bin4(float4 a, float4 b) {
    return make_float4(bin_t<OP>(a.x, b.x), bin_t<OP>(a.y, b.y), bin_t<OP>(a.z, b.z),
                       bin_t<OP>(a.w, b.w));
}

template <int ACT>
__device__ __forceinline__ float4 act4(float4 t) {
    return make_float4(act<ACT>(t.x), act<ACT>(t.y), act<ACT>(t.z), act<ACT>(t.w));
}

// Grid for a flat streaming kernel: enough workgroups to fill 256 CUs
// several times over, each thread then strides through the rest.
inline unsigned stream_grid(size_t n4) {
    size_t b = (n4 + kBlock - 1) / kBlock;
    const size_t cap = 256 * 16;
    return static_cast<unsigned>(b < 1 ? 1 : (b > cap ? cap : b));
}

// -------------------------------------------------------------- binary

__global__ __launch_bounds__(kBlock) void k_binary_scalar(const float *x, const float *y, float *z,
                                                          size_t n, int op) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride)
        z[i] = bin(op, x[i], y[i]);
}

// ------------------------------------------------------------ broadcast

__global__ __launch_bounds__(kBlock) void k_bcast_scalar(const float *x, const float *y, float *z,
                                                         size_t m, size_t n, int op, int row_mode) {
    const size_t total = m * n;
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
        const size_t r = i / n;
        const size_t c = i - r * n;
        z[i] = bin(op, x[i], row_mode ? y[c] : y[r]);
    }
}

// --------------------------------------------------------------- scalar

__global__ __launch_bounds__(kBlock) void k_scalar_scalar(const float *x, float v, float *z, size_t n,
                                                          int op) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride)
        z[i] = bin(op, x[i], v);
}

// ---------------------------------------------------------------- unary

template <int ACT>
__global__ __launch_bounds__(kBlock) void k_unary_scalar(const float *x, float *z, size_t n) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride)
        z[i] = act<ACT>(x[i]);
}

// Functors of the streaming maps (k_map4 / k_zip4 / k_rowmap4).
template <int OP>
struct BinF {
    __device__ float operator()(float a, float b) const { return bin_t<OP>(a, b); }
};
template <int OP>
struct ScalarF {
    float v;
    __device__ float operator()(float a) const { return bin_t<OP>(a, v); }
};
template <int ACT>
struct ActF {
    __device__ float operator()(float t) const { return act<ACT>(t); }
};
// ---------------------------------------------------- flat row maps
//
// Row-structured maps over rows that are no multiple of four floats, or too
// short for k_rowmap4's 256-column tiles: the matrix is read as one run of
// aligned float4s, and a float4's row and column come from its index by a
// multiplication with the row length's precomputed reciprocal.  A float4 that
// runs past its row's end takes the next row's operands for the rest (rows
// are at least four floats long, so there is one such end at most).
// Measured: row broadcast over [3001, 1003] 6.9 -> 5.6 us (a 64-bit division and
// dword accesses per element before), [2396, 55] 4.2 -> 3.9 us (a launch).

// Division of 32-bit numbers by an invariant d >= 1: Granlund and Montgomery,
// "Division by invariant integers using multiplication" (1994), figure 4.1.
struct FastDiv {
    unsigned mul, sh1, sh2;
    __device__ unsigned operator()(unsigned e) const {
        const unsigned t = __umulhi(mul, e);
        return (t + ((e - t) >> sh1)) >> sh2;
    }
};
inline FastDiv fast_div(unsigned d) {
    unsigned l = 0;
    while (l < 32 && (1ull << l) < d) ++l;
    const unsigned long long m = ((1ull << 32) * ((1ull << l) - d)) / d + 1;
    return FastDiv{static_cast<unsigned>(m), l < 1 ? l : 1u, l < 1 ? 0u : l - 1};
}

// y[c .. c+3] of an n-float row, wrapping to y[0 ..] past its end (c < n, n >= 4).
__device__ __forceinline__ float4 wrap4(const float *__restrict__ y, unsigned c, unsigned n) {
    const unsigned off = c < n - 4 ? c : n - 4, d = c - off;
    const float4 v = ld4_any<false>(y + off), h = ld4_any<false>(y);
    float4 o;
    o.x = d == 0 ? v.x : d == 1 ? v.y : d == 2 ? v.z : v.w;
    o.y = d == 0 ? v.y : d == 1 ? v.z : d == 2 ? v.w : h.x;
    o.z = d == 0 ? v.z : d == 1 ? v.w : d == 2 ? h.x : h.y;
    o.w = d == 0 ? v.w : d == 1 ? h.x : d == 2 ? h.y : h.z;
    return o;
}

// f.flat(v, r, c, m, n): the output float4 for the elements at (r, c ..),
// f.one(v, r, c): one element.
template <class F, bool AL>
__global__ __launch_bounds__(kBlock) void k_flatmap4(F f, const float *x, float *z, unsigned total, unsigned m,
                                                     unsigned n, FastDiv by_n) {
    const size_t i = stream_vec();
    const unsigned n4 = total / 4;
    if (i < n4) {
        const unsigned e = 4 * static_cast<unsigned>(i), r = by_n(e);
        st4_any_stream<AL>(z + e, f.flat(ld4_any_stream<AL>(x + e), r, e - r * n, m, n));
    } else if (i == n4) {
        for (unsigned j = 4 * n4; j < total; ++j) {
            const unsigned r = by_n(j);
            z[j] = f.one(x[j], r, j - r * n);
        }
    }
}

// Whether the flat map takes an [m, n] row map: 32-bit element numbers, and
// rows that k_rowmap4 does not take (`rows4`: n a multiple of 4, everything
// 16-byte aligned) or leaves more than a fifth of its lanes idle on.
// Measured at [m, n], flat / row tiles (us): affine forward [60000, 32] 4.7 /
// 14.2, [3000, 520] 4.3 / 5.2, [4096, 320] 4.1 / 4.3, [7000, 480] 6.7 / 6.6,
// [8192, 8192] 87.5 / 82.5 (its operands cross from L2 once per wave).
inline bool use_flatmap(size_t m, size_t n, bool rows4) {
    if (n < 4 || m > 0xfffffc00u / n) return false;
    const size_t n4 = n / 4, lanes = (n4 + kWave - 1) / kWave * kWave;
    return !rows4 || n4 * 5 < lanes * 4;
}

template <class F>
int run_flatmap(const F &f, const float *x, float *z, size_t m, size_t n, hipStream_t s) {
    const unsigned total = static_cast<unsigned>(m * n), g = map4_grid(total);
    const FastDiv d = fast_div(static_cast<unsigned>(n));
    if (aligned16(x) && aligned16(z))
        hipLaunchKernelGGL((k_flatmap4<F, true>), dim3(g), dim3(kBlock), 0, s, f, x, z, total, static_cast<unsigned>(m),
                           static_cast<unsigned>(n), d);
    else
        hipLaunchKernelGGL((k_flatmap4<F, false>), dim3(g), dim3(kBlock), 0, s, f, x, z, total, static_cast<unsigned>(m),
                           static_cast<unsigned>(n), d);
    return launch_status();
}

// z[i,j] = x[i,j] op y[j]
template <int OP>
struct RowBcastF {
    const float *y;
    __device__ float4 operator()(float4 v, unsigned, size_t j4) const { return bin4<OP>(v, ld4(y + 4 * j4)); }
    __device__ float4 flat(float4 v, unsigned, unsigned c, unsigned, unsigned n) const {
        return bin4<OP>(v, wrap4(y, c, n));
    }
    __device__ float one(float v, unsigned, unsigned c) const { return bin_t<OP>(v, y[c]); }
};
// z[i,j] = x[i,j] op y[i]
template <int OP>
struct ColBcastF {
    const float *y;
    __device__ float4 operator()(float4 v, unsigned row, size_t) const {
        const float c = y[row];
        return bin4<OP>(v, make_float4(c, c, c, c));
    }
    __device__ float4 flat(float4 v, unsigned r, unsigned c, unsigned m, unsigned n) const {
        const float a = y[r], b = y[r + 1 < m ? r + 1 : r];
        return bin4<OP>(v, make_float4(a, c + 1 < n ? a : b, c + 2 < n ? a : b, c + 3 < n ? a : b));
    }
    __device__ float one(float v, unsigned r, unsigned) const { return bin_t<OP>(v, y[r]); }
};
// y = act(x*scale[j] + bias[j]): product and sum rounded separately
template <int ACT>
struct AffineF {
    const float *scale, *bias;
    __device__ float4 operator()(float4 v, unsigned, size_t j4) const {
        return apply(v, ld4(scale + 4 * j4), ld4(bias + 4 * j4));
    }
    __device__ float4 flat(float4 v, unsigned, unsigned c, unsigned, unsigned n) const {
        return apply(v, wrap4(scale, c, n), wrap4(bias, c, n));
    }
    __device__ float one(float v, unsigned, unsigned c) const {
        float t = v * scale[c];
        t = t + bias[c];
        return act<ACT>(t);
    }
    __device__ static float4 apply(float4 v, float4 sc, float4 b) {
        float4 t;
        t.x = v.x * sc.x; t.y = v.y * sc.y; t.z = v.z * sc.z; t.w = v.w * sc.w;
        t.x = t.x + b.x; t.y = t.y + b.y; t.z = t.z + b.z; t.w = t.w + b.w;
        return act4<ACT>(t);
    }
};
// dx = dy * act'(y), the derivative factor from the saved output
template <int ACT>
struct ActBwdF {
    __device__ float operator()(float y, float g) const { return g * dact<ACT>(y); }
};
// w - g*lr, two roundings
struct SgdF {
    float lr;
    __device__ float operator()(float w, float g) const {
        const float t = g * lr;
        return w - t;
    }
};

// ------------------------------------------------------ affine forward

template <int ACT>
__global__ __launch_bounds__(kBlock) void k_affine_fwd_scalar(const float *x, const float *scale,
                                                              const float *bias, float *y, size_t m,
                                                              size_t n) {
    const size_t total = m * n;
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
        const size_t c = i % n;
        float t = x[i] * scale[c];
        t = t + bias[c];
        y[i] = act<ACT>(t);
    }
}

// ----------------------------------------------------- affine backward

constexpr unsigned kAffGroups = 32;  // groups of chunks of one tile (512 chunks at most)

// dz = dy*act'(y); dx = dz*scale[j]; dscale[j] = sum_i dz*x; dbias[j] = sum_i dz.
// A 256-thread workgroup takes a tile of 4 G columns (G lanes x float4) and a
// chunk of rows; its 256 / G lane groups take interleaved rows, UNR of them
// in flight, and meet in LDS pairwise, as do the chunks' partials in eights
// (all one after the other, dbias of [40, 16] was 1.2e-7 from 64 bits and of
// [700, 4096] 1.3e-7; 8e-8 and 1.0e-7 so).  The chunks of a tile are adjacent
// in launch order, so early tiles' combines overlap later tiles' streaming; the
// last workgroup of a tile combines them in chunk order, beyond 32 chunks in
// two levels (groups of kPartGroup).  AL: 16-byte aligned rows (G = 64 only);
// otherwise dword-aligned accesses, the last lane of a row reading its last
// four columns and keeping its own (n >= 4).  [6848, 83] backward 43 -> 7.9 us
// (dword accesses, and one workgroup summing 428 partials, before);
// [8192, 256] 50 -> 13.5 us.
constexpr int kAffTile = 256;  // stride of a tile's partials

template <int ACT, bool AL, int G, int UNR>
__global__ __launch_bounds__(kBlock) void k_affine_bwd(const float *__restrict__ x, const float *__restrict__ scale,
                                                       const float *__restrict__ y, const float *__restrict__ dy,
                                                       float *__restrict__ dx, float *__restrict__ dscale,
                                                       float *__restrict__ dbias, size_t m, size_t n, unsigned chunks,
                                                       size_t rows_per_chunk, float *__restrict__ part,
                                                       float *__restrict__ tops, unsigned *__restrict__ counters) {
    constexpr int NS = kBlock / G, TW = 4 * G;
    __shared__ float lds_s[NS][TW];
    __shared__ float lds_b[NS][TW];
    __shared__ int flag;
    const unsigned tile = blockIdx.x / chunks, chunk = blockIdx.x - tile * chunks;
    const int tid = threadIdx.x, lane = tid % G, g = tid / G;
    const size_t r0 = static_cast<size_t>(chunk) * rows_per_chunk;
    const size_t r1 = r0 + rows_per_chunk < m ? r0 + rows_per_chunk : m;
    const size_t col = static_cast<size_t>(tile) * TW + lane * 4;
    const size_t pos = AL || col + 4 <= n ? col : n - 4;
    const int d = col < n ? static_cast<int>(col - pos) : 4;  // columns pos .. pos + d - 1 are another lane's
    float as[4] = {0, 0, 0, 0}, ab[4] = {0, 0, 0, 0};
    if (d < 4) {
        const float4 sc = ld4_any<AL>(scale + pos);
        size_t r = r0 + g;
        auto body = [&](size_t rr, float4 xv, float4 yv, float4 gv) {
            float4 dz;
            dz.x = gv.x * dact<ACT>(yv.x); dz.y = gv.y * dact<ACT>(yv.y);
            dz.z = gv.z * dact<ACT>(yv.z); dz.w = gv.w * dact<ACT>(yv.w);
            float4 o;
            o.x = dz.x * sc.x; o.y = dz.y * sc.y; o.z = dz.z * sc.z; o.w = dz.w * sc.w;
            float *p = dx + rr * n + pos;
            if (AL || d == 0) {
                st4_any_stream<AL>(p, o);
            } else {
                if (d <= 1) p[1] = o.y;
                if (d <= 2) p[2] = o.z;
                p[3] = o.w;
            }
            const float p0 = dz.x * xv.x, p1 = dz.y * xv.y, p2 = dz.z * xv.z, p3 = dz.w * xv.w;
            as[0] = as[0] + p0; as[1] = as[1] + p1; as[2] = as[2] + p2; as[3] = as[3] + p3;
            ab[0] = ab[0] + dz.x; ab[1] = ab[1] + dz.y; ab[2] = ab[2] + dz.z; ab[3] = ab[3] + dz.w;
        };
        for (; r < r1; r += UNR * NS) {
            float4 xv[UNR], yv[UNR], gv[UNR];
#pragma unroll
            for (int u = 0; u < UNR; ++u) {  // rows past the chunk's end re-read its last one
                const size_t o = (UNR == 1 || r + u * NS < r1 ? r + u * NS : r1 - 1) * n + pos;
                xv[u] = ld4_any_stream<AL>(x + o);
                yv[u] = ld4_any_stream<AL>(y + o);
                gv[u] = ld4_any_stream<AL>(dy + o);
            }
            if constexpr (UNR > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < UNR; ++u)
                if (UNR == 1 || r + u * NS < r1) body(r + u * NS, xv[u], yv[u], gv[u]);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (d < 4 && c >= d) {
            lds_s[g][lane * 4 + c - d] = as[c];
            lds_b[g][lane * 4 + c - d] = ab[c];
        }
    }
    __syncthreads();
    const size_t oc = static_cast<size_t>(tile) * TW + tid;
    const bool put = tid < TW && oc < n;  // these threads own one column each from here
    float ms = 0.0f, mb = 0.0f;
    if (put) {
        ms = combine_pairwise<SumOp, NS>(&lds_s[0][tid], TW);
        mb = combine_pairwise<SumOp, NS>(&lds_b[0][tid], TW);
    }
    if (chunks == 1) {
        if (put) {
            dscale[oc] = ms;
            dbias[oc] = mb;
        }
        return;
    }
    // the sum of `count` pairs of partials, eight at a time in flight and
    // pairwise
    auto sum = [&](const float *p, unsigned count) {
        ms = 0.0f;
        mb = 0.0f;
        for (unsigned c0 = 0; c0 < count; c0 += 8) {
            float va[8], vb[8];
#pragma unroll
            for (unsigned u = 0; u < 8; ++u) {
                const bool in = c0 + u < count;
                va[u] = in ? ld_dev(&p[((c0 + u) * 2 + 0) * kAffTile + tid]) : 0.0f;
                vb[u] = in ? ld_dev(&p[((c0 + u) * 2 + 1) * kAffTile + tid]) : 0.0f;
            }
            ms = ms + (((va[0] + va[1]) + (va[2] + va[3])) + ((va[4] + va[5]) + (va[6] + va[7])));
            mb = mb + (((vb[0] + vb[1]) + (vb[2] + vb[3])) + ((vb[4] + vb[5]) + (vb[6] + vb[7])));
        }
    };
    float *pt = part + static_cast<size_t>(tile) * chunks * 2 * kAffTile;
    if (put) {
        st_dev(&pt[(static_cast<size_t>(chunk) * 2 + 0) * kAffTile + tid], ms);
        st_dev(&pt[(static_cast<size_t>(chunk) * 2 + 1) * kAffTile + tid], mb);
    }
    if (chunks <= 2 * kPartGroup) {
        if (!last_block_ticket(ctr(counters, tile), chunks, &flag)) return;
        if (put) sum(pt, chunks);
    } else {
        const unsigned groups = (chunks + kPartGroup - 1) / kPartGroup, q = chunk / kPartGroup;
        const unsigned size = (q + 1) * kPartGroup <= chunks ? kPartGroup : chunks - q * kPartGroup;
        unsigned *cg = ctr(counters, static_cast<size_t>(tile) * (kAffGroups + 1));
        float *tp = tops + static_cast<size_t>(tile) * kAffGroups * 2 * kAffTile;
        if (!last_block_ticket(ctr(cg, q), size, &flag)) return;
        if (put) {
            sum(pt + static_cast<size_t>(q) * kPartGroup * 2 * kAffTile, size);
            st_dev(&tp[(q * 2 + 0) * kAffTile + tid], ms);
            st_dev(&tp[(q * 2 + 1) * kAffTile + tid], mb);
        }
        if (!last_block_ticket(ctr(cg, kAffGroups), groups, &flag)) return;
        if (put) sum(tp, groups);
    }
    if (put) {
        dscale[oc] = ms;
        dbias[oc] = mb;
    }
}

// Rows of fewer than four floats: thread t of a chunk's workgroup takes
// column t % n of every 256 / n-th row; the last workgroup adds the at most
// 256 chunks' partials, a chunk per thread.
template <int ACT>
__global__ __launch_bounds__(kBlock) void k_affine_bwd_few(const float *__restrict__ x, const float *__restrict__ scale,
                                                           const float *__restrict__ y, const float *__restrict__ dy,
                                                           float *__restrict__ dx, float *__restrict__ dscale,
                                                           float *__restrict__ dbias, size_t m, unsigned n,
                                                           unsigned chunks, size_t rows_per_chunk,
                                                           float *__restrict__ part, unsigned *__restrict__ counters) {
    __shared__ float lds[kWavesPerBlock];
    __shared__ int flag;
    const unsigned rows = kBlock / n, c = threadIdx.x % n, g = threadIdx.x / n;
    const size_t r0 = blockIdx.x * rows_per_chunk, r1 = r0 + rows_per_chunk < m ? r0 + rows_per_chunk : m;
    float ms = 0.0f, mb = 0.0f;
    if (g < rows) {
        const float sc = scale[c];
        for (size_t r = r0 + g; r < r1; r += rows) {
            const size_t o = r * n + c;
            const float dz = dy[o] * dact<ACT>(y[o]);
            const float p = dz * x[o];
            dx[o] = dz * sc;
            ms = ms + p;
            mb = mb + dz;
        }
    }
    for (unsigned j = 0; j < n; ++j) {
        const float s = block_reduce<SumOp, kBlock>(c == j && g < rows ? ms : 0.0f, lds);
        const float b = block_reduce<SumOp, kBlock>(c == j && g < rows ? mb : 0.0f, lds);
        if (threadIdx.x != 0) continue;
        if (chunks == 1) {
            dscale[j] = s;
            dbias[j] = b;
        } else {
            st_dev(&part[(j * 2 + 0) * kBlock + blockIdx.x], s);
            st_dev(&part[(j * 2 + 1) * kBlock + blockIdx.x], b);
        }
    }
    if (chunks == 1 || !last_block_ticket2<kAffGroups>(counters, chunks, blockIdx.x, &flag)) return;
    for (unsigned j = 0; j < n; ++j) {
        const bool in = threadIdx.x < chunks;
        const float s = block_reduce<SumOp, kBlock>(in ? ld_dev(&part[(j * 2 + 0) * kBlock + threadIdx.x]) : 0.0f, lds);
        const float b = block_reduce<SumOp, kBlock>(in ? ld_dev(&part[(j * 2 + 1) * kBlock + threadIdx.x]) : 0.0f, lds);
        if (threadIdx.x == 0) {
            dscale[j] = s;
            dbias[j] = b;
        }
    }
}

// ------------------------------------------------------------------ sgd

// w = w - g*lr, two roundings (matrix_t::sub of ScalarOp::mul).
__global__ __launch_bounds__(kBlock) void k_act_bwd_scalar(const float *y, const float *dy, float *dx, size_t n,
                                                            int act) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
        const float yy = y[i];
        const float d = act == CXM_ACT_RELU ? dact<CXM_ACT_RELU>(yy)
                                            : (act == CXM_ACT_SIGMOID ? dact<CXM_ACT_SIGMOID>(yy) : dact<CXM_ACT_TANH>(yy));
        dx[i] = dy[i] * d;
    }
}

__global__ __launch_bounds__(kBlock) void k_sgd_scalar(float *w, const float *g, float lr, size_t n) {
    const size_t stride = static_cast<size_t>(gridDim.x) * kBlock;
    for (size_t i = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
        const float t = g[i] * lr;
        w[i] = w[i] - t;
    }
}

// ----------------------------------------------------------------- host

inline hipStream_t hs(cxm_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

template <template <int> class L, class... A>
int dispatch_op(int op, A... a) {
    switch (op) {
        case CXM_OP_ADD: return L<CXM_OP_ADD>::run(a...);
        case CXM_OP_SUB: return L<CXM_OP_SUB>::run(a...);
        case CXM_OP_MUL: return L<CXM_OP_MUL>::run(a...);
        case CXM_OP_DIV: return L<CXM_OP_DIV>::run(a...);
        case CXM_OP_MAX: return L<CXM_OP_MAX>::run(a...);
        case CXM_OP_MIN: return L<CXM_OP_MIN>::run(a...);
        case CXM_OP_POW: return L<CXM_OP_POW>::run(a...);
        default: return CXM_E_INVALID;
    }
}

template <int OP>
struct BinaryL {
    static int run(const float *x, const float *y, float *z, size_t n, hipStream_t s) {
        const unsigned g = map4_grid(n);
        if (!g) return CXM_E_TOO_LARGE;
        hipLaunchKernelGGL(k_zip4<BinF<OP>>, dim3(g), dim3(kBlock), 0, s, BinF<OP>{}, x, y, z, n);
        return launch_status();
    }
};

template <int OP>
struct ScalarL {
    static int run(const float *x, float v, float *z, size_t n, hipStream_t s) {
        const unsigned g = map4_grid(n);
        if (!g) return CXM_E_TOO_LARGE;
        hipLaunchKernelGGL(k_map4<ScalarF<OP>>, dim3(g), dim3(kBlock), 0, s, ScalarF<OP>{v}, x, z, n);
        return launch_status();
    }
};

template <int OP>
struct BcastL {
    static int run(const float *x, const float *y, float *z, size_t m, size_t n, int row_mode,
                   hipStream_t s) {
        unsigned grid, tpr;
        if (!rowmap4_grid(m, n / 4, &grid, &tpr)) return CXM_E_TOO_LARGE;
        if (row_mode)
            hipLaunchKernelGGL(k_rowmap4<RowBcastF<OP>>, dim3(grid), dim3(kBlock), 0, s, RowBcastF<OP>{y}, x, z,
                               m, n / 4, tpr);
        else
            hipLaunchKernelGGL(k_rowmap4<ColBcastF<OP>>, dim3(grid), dim3(kBlock), 0, s, ColBcastF<OP>{y}, x, z,
                               m, n / 4, tpr);
        return launch_status();
    }
};

template <int OP>
struct BcastFlatL {
    static int run(const float *x, const float *y, float *z, size_t m, size_t n, int row_mode, hipStream_t s) {
        if (row_mode) return run_flatmap(RowBcastF<OP>{y}, x, z, m, n, s);
        return run_flatmap(ColBcastF<OP>{y}, x, z, m, n, s);
    }
};

int bcast(const float *x, const float *y, float *z, size_t m, size_t n, int op, int row_mode,
          cxm_stream_t s) {
    if (!x || !y || !z || op < CXM_OP_ADD || op > CXM_OP_DIV) return CXM_E_INVALID;
    if (m == 0 || n == 0) return CXM_OK;
    const bool rows4 = n % 4 == 0 && aligned16(x) && aligned16(z) && (!row_mode || aligned16(y));
    if (use_flatmap(m, n, rows4)) return dispatch_op<BcastFlatL>(op, x, y, z, m, n, row_mode, hs(s));
    if (rows4) return dispatch_op<BcastL>(op, x, y, z, m, n, row_mode, hs(s));
    hipLaunchKernelGGL(k_bcast_scalar, dim3(stream_grid((m * n + 3) / 4)), dim3(kBlock), 0, hs(s), x,
                       y, z, m, n, op, row_mode);
    return launch_status();
}

template <int ACT>
int unary_t(const float *x, float *z, size_t n, hipStream_t s) {
    if (aligned16(x) && aligned16(z)) {
        const unsigned g = map4_grid(n);
        if (!g) return CXM_E_TOO_LARGE;
        hipLaunchKernelGGL(k_map4<ActF<ACT>>, dim3(g), dim3(kBlock), 0, s, ActF<ACT>{}, x, z, n);
    } else {
        hipLaunchKernelGGL(k_unary_scalar<ACT>, dim3(stream_grid((n + 3) / 4)), dim3(kBlock), 0, s, x, z, n);
    }
    return launch_status();
}

template <int ACT>
int affine_fwd_t(const float *x, const float *scale, const float *bias, float *y, size_t m,
                 size_t n, hipStream_t s) {
    unsigned grid, tpr;
    const bool rows4 = n % 4 == 0 && aligned16(x) && aligned16(scale) && aligned16(bias) && aligned16(y);
    if (use_flatmap(m, n, rows4)) return run_flatmap(AffineF<ACT>{scale, bias}, x, y, m, n, s);
    if (rows4 && rowmap4_grid(m, n / 4, &grid, &tpr)) {
        hipLaunchKernelGGL(k_rowmap4<AffineF<ACT>>, dim3(grid), dim3(kBlock), 0, s, AffineF<ACT>{scale, bias},
                           x, y, m, n / 4, tpr);
    } else {
        hipLaunchKernelGGL(k_affine_fwd_scalar<ACT>, dim3(stream_grid((m * n + 3) / 4)), dim3(kBlock), 0,
                           s, x, scale, bias, y, m, n);
    }
    return launch_status();
}

// Row chunks per column tile and launch order.  Measured on gfx950 at 256 MiB
// per operand, sigmoid: 512 workgroups of 4 waves (two per CU, each
// streaming a few hundred rows), one row of loads per wave in flight and
// the chunks of a tile adjacent in launch order reach 6.5 TB/s at
// [8192, 8192] and 6.7 TB/s at [1024, 65536].  Deeper unrolling (2 or 4
// rows of loads per wave, with or without a scheduling barrier that keeps
// them together), 2048 shorter workgroups, 384 workgroups (CUs unevenly
// loaded) and 16-wave workgroups were all slower, by 5-25%.
// Few rows per lane group (at most kAffFew) have several rows of loads in
// flight where rows are narrow (four: [20000, 16] 8.7 -> 7.7 us, [8000, 96] 9.3
// -> 7.9) or ragged (two: [3001, 1003] 16.0 -> 15.0): there the serial round
// trips count.  Wide aligned rows keep one ([4000, 1000] 16.9 us with one,
// 18.3 with four).
constexpr size_t kAffFew = 16;

template <int ACT, bool AL, int G>
int affine_bwd_launch(const float *x, const float *scale, const float *y, const float *dy, float *dx, float *dscale,
                      float *dbias, size_t m, size_t n, cxm_stream_t st) {
    constexpr size_t NS = kBlock / G, TW = 4 * G;
    const size_t ntiles = (n + TW - 1) / TW;
    size_t chunks = 512 / ntiles;  // one more workgroup than 512 would be a round of its own
    const size_t max_chunks = (m + 4 * NS - 1) / (4 * NS);  // at least four rows per lane group
    if (chunks > max_chunks) chunks = max_chunks;
    if (chunks < 1) chunks = 1;
    size_t rpc = (m + chunks - 1) / chunks;
    rpc = (rpc + NS - 1) / NS * NS;
    chunks = (m + rpc - 1) / rpc;
    if (ntiles * chunks > 0x7fffffffu) return CXM_E_TOO_LARGE;
    float *part = nullptr, *tops = nullptr;
    unsigned *counters = nullptr;
    if (chunks > 1) {
        Workspace ws;
        const bool two = chunks > 2 * kPartGroup;
        int rc = get_workspace(st, two ? ntiles * (kAffGroups + 1) : ntiles,
                               ntiles * (chunks + (two ? kAffGroups : 0)) * 2 * kAffTile * sizeof(float), &ws);
        if (rc) return rc;
        part = static_cast<float *>(ws.scratch);
        tops = part + ntiles * chunks * 2 * kAffTile;
        counters = ws.counters;
    }
    const dim3 grid(static_cast<unsigned>(ntiles * chunks));
    const unsigned nc = static_cast<unsigned>(chunks);
    constexpr int kUnr = G < kWave ? 4 : AL ? 1 : 2;
    if (kUnr > 1 && rpc <= kAffFew * NS)
        hipLaunchKernelGGL((k_affine_bwd<ACT, AL, G, kUnr>), grid, dim3(kBlock), 0, hs(st), x, scale, y, dy, dx, dscale,
                           dbias, m, n, nc, rpc, part, tops, counters);
    else
        hipLaunchKernelGGL((k_affine_bwd<ACT, AL, G, 1>), grid, dim3(kBlock), 0, hs(st), x, scale, y, dy, dx, dscale,
                           dbias, m, n, nc, rpc, part, tops, counters);
    return launch_status();
}

template <int ACT>
int affine_bwd_t(const float *x, const float *scale, const float *y, const float *dy, float *dx,
                 float *dscale, float *dbias, size_t m, size_t n, cxm_stream_t st) {
    if (n < 4) {
        size_t chunks = (m + 1023) / 1024 < kBlock ? (m + 1023) / 1024 : kBlock;
        const size_t rpc = (m + chunks - 1) / chunks;
        chunks = (m + rpc - 1) / rpc;
        Workspace ws{};
        if (chunks > 1) {
            const int rc = get_workspace(st, kAffGroups + 1, 6 * kBlock * sizeof(float), &ws);
            if (rc) return rc;
        }
        hipLaunchKernelGGL(k_affine_bwd_few<ACT>, dim3(static_cast<unsigned>(chunks)), dim3(kBlock), 0, hs(st), x, scale,
                           y, dy, dx, dscale, dbias, m, static_cast<unsigned>(n), static_cast<unsigned>(chunks), rpc,
                           static_cast<float *>(ws.scratch), ws.counters);
        return launch_status();
    }
    // the fewest lanes whose float4s cover a row, up to a wave
    const size_t v4 = (n + 3) / 4;
    if (v4 <= 8) return affine_bwd_launch<ACT, false, 8>(x, scale, y, dy, dx, dscale, dbias, m, n, st);
    if (v4 <= 16) return affine_bwd_launch<ACT, false, 16>(x, scale, y, dy, dx, dscale, dbias, m, n, st);
    if (v4 <= 32) return affine_bwd_launch<ACT, false, 32>(x, scale, y, dy, dx, dscale, dbias, m, n, st);
    if (n % 4 == 0 && aligned16(x) && aligned16(scale) && aligned16(y) && aligned16(dy) && aligned16(dx))
        return affine_bwd_launch<ACT, true, 64>(x, scale, y, dy, dx, dscale, dbias, m, n, st);
    return affine_bwd_launch<ACT, false, 64>(x, scale, y, dy, dx, dscale, dbias, m, n, st);
}

// ------------------------------------------------- sum / mean backward

// dx[o, d, i] = g(dz[o, i]) over dx as row-major [outer, dim, inner], with
// g(v) = v for a sum and v / dim for a mean.  One float4 of dx per thread
// (the grid of k_map4).  MODE 0: inner == 1 and dim % 4 == 0, so a float4
// lies in one row o and repeats dz[o]; MODE 1: inner % 4 == 0, a float4 is
// four consecutive inner indices of one (o, d), read as a float4 of dz;
// MODE 2: any shape or alignment, element by element.
template <bool MEAN, int MODE>
__global__ __launch_bounds__(kBlock) void k_sum_bwd(const float *__restrict__ dz, float *__restrict__ dx, size_t dim,
                                                    size_t inner, size_t n, float dimf) {
    const size_t t = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x;
    const size_t e = 4 * t;
    if (e >= n) return;
    auto g = [dimf](float v) { return MEAN ? v / dimf : v; };
    if constexpr (MODE == 0) {
        const float v = g(dz[e / dim]);
        st4_stream(dx + e, make_float4(v, v, v, v));
    } else if constexpr (MODE == 1) {
        const size_t slab = dim * inner;
        const size_t o = e / slab, i = e % inner;
        const float4 v = ld4(dz + o * inner + i);
        st4_stream(dx + e, make_float4(g(v.x), g(v.y), g(v.z), g(v.w)));
    } else {
        const size_t slab = dim * inner;
        for (size_t k = e; k < e + 4 && k < n; ++k) dx[k] = g(dz[(k / slab) * inner + k % inner]);
    }
}

template <bool MEAN>
int sum_bwd_t(const float *dz, float *dx, size_t outer, size_t dim, size_t inner, hipStream_t s) {
    const size_t n = outer * dim * inner;
    const unsigned grid = map4_grid(n + 3);
    if (!grid) return CXM_E_TOO_LARGE;
    const float dimf = static_cast<float>(dim);
    if (aligned16(dx) && inner == 1 && dim % 4 == 0)
        hipLaunchKernelGGL((k_sum_bwd<MEAN, 0>), dim3(grid), dim3(kBlock), 0, s, dz, dx, dim, inner, n, dimf);
    else if (aligned16(dx) && aligned16(dz) && inner % 4 == 0)
        hipLaunchKernelGGL((k_sum_bwd<MEAN, 1>), dim3(grid), dim3(kBlock), 0, s, dz, dx, dim, inner, n, dimf);
    else
        hipLaunchKernelGGL((k_sum_bwd<MEAN, 2>), dim3(grid), dim3(kBlock), 0, s, dz, dx, dim, inner, n, dimf);
    return launch_status();
}

}  // namespace
}  // namespace cxm

using namespace cxm;

extern "C" {

int cxm_binary_f32(const float *x, const float *y, float *z, size_t n, int op, cxm_stream_t s) {
    if (!x || !y || !z || op < CXM_OP_ADD || op > CXM_OP_POW) return CXM_E_INVALID;
    if (n == 0) return CXM_OK;
    if (aligned16(x) && aligned16(y) && aligned16(z)) return dispatch_op<BinaryL>(op, x, y, z, n, hs(s));
    hipLaunchKernelGGL(k_binary_scalar, dim3(stream_grid((n + 3) / 4)), dim3(kBlock), 0, hs(s), x, y, z,
                       n, op);
    return launch_status();
}

int cxm_bcast_row_f32(const float *x, const float *y, float *z, size_t m, size_t n, int op,
                      cxm_stream_t s) {
    return bcast(x, y, z, m, n, op, 1, s);
}

int cxm_bcast_col_f32(const float *x, const float *y, float *z, size_t m, size_t n, int op,
                      cxm_stream_t s) {
    return bcast(x, y, z, m, n, op, 0, s);
}

int cxm_scalar_f32(const float *x, float value, float *z, size_t n, int op, cxm_stream_t s) {
    if (!x || !z || op < CXM_OP_ADD || op > CXM_OP_POW) return CXM_E_INVALID;
    if (n == 0) return CXM_OK;
    if (aligned16(x) && aligned16(z)) return dispatch_op<ScalarL>(op, x, value, z, n, hs(s));
    hipLaunchKernelGGL(k_scalar_scalar, dim3(stream_grid((n + 3) / 4)), dim3(kBlock), 0, hs(s), x, value,
                       z, n, op);
    return launch_status();
}

int cxm_unary_f32(const float *x, float *z, size_t n, int act, cxm_stream_t s) {
    if (!x || !z) return CXM_E_INVALID;
    if (n == 0) return CXM_OK;
    switch (act) {
        case CXM_ACT_RELU: return unary_t<CXM_ACT_RELU>(x, z, n, hs(s));
        case CXM_ACT_SIGMOID: return unary_t<CXM_ACT_SIGMOID>(x, z, n, hs(s));
        case CXM_ACT_TANH: return unary_t<CXM_ACT_TANH>(x, z, n, hs(s));
        case CXM_ACT_EXP: return unary_t<CXM_ACT_EXP>(x, z, n, hs(s));
        default: return CXM_E_INVALID;
    }
}

int cxm_affine_act_fwd_f32(const float *x, const float *scale, const float *bias, float *y,
                           size_t m, size_t n, int act, cxm_stream_t s) {
    if (!x || !scale || !bias || !y) return CXM_E_INVALID;
    if (m == 0 || n == 0) return CXM_OK;
    switch (act) {
        case CXM_ACT_NONE: return affine_fwd_t<CXM_ACT_NONE>(x, scale, bias, y, m, n, hs(s));
        case CXM_ACT_RELU: return affine_fwd_t<CXM_ACT_RELU>(x, scale, bias, y, m, n, hs(s));
        case CXM_ACT_SIGMOID: return affine_fwd_t<CXM_ACT_SIGMOID>(x, scale, bias, y, m, n, hs(s));
        case CXM_ACT_TANH: return affine_fwd_t<CXM_ACT_TANH>(x, scale, bias, y, m, n, hs(s));
        default: return CXM_E_INVALID;
    }
}

int cxm_affine_act_bwd_f32(const float *x, const float *scale, const float *y, const float *dy,
                           float *dx, float *dscale, float *dbias, size_t m, size_t n, int act,
                           cxm_stream_t s) {
    if (!x || !scale || !y || !dy || !dx || !dscale || !dbias) return CXM_E_INVALID;
    if (n == 0) return CXM_OK;
    if (m == 0) return CXM_E_INVALID;  // column sums over zero rows are undefined in the reference
    switch (act) {
        case CXM_ACT_NONE:
            return affine_bwd_t<CXM_ACT_NONE>(x, scale, y, dy, dx, dscale, dbias, m, n, s);
        case CXM_ACT_RELU:
            return affine_bwd_t<CXM_ACT_RELU>(x, scale, y, dy, dx, dscale, dbias, m, n, s);
        case CXM_ACT_SIGMOID:
            return affine_bwd_t<CXM_ACT_SIGMOID>(x, scale, y, dy, dx, dscale, dbias, m, n, s);
        case CXM_ACT_TANH:
            return affine_bwd_t<CXM_ACT_TANH>(x, scale, y, dy, dx, dscale, dbias, m, n, s);
        default: return CXM_E_INVALID;
    }
}

int cxm_act_bwd_f32(const float *y, const float *dy, float *dx, size_t n, int act, cxm_stream_t s) {
    if (!y || !dy || !dx || act < CXM_ACT_RELU || act > CXM_ACT_TANH) return CXM_E_INVALID;
    if (n == 0) return CXM_OK;
    if (!(aligned16(y) && aligned16(dy) && aligned16(dx))) {
        hipLaunchKernelGGL(k_act_bwd_scalar, dim3(stream_grid((n + 3) / 4)), dim3(kBlock), 0, hs(s), y, dy, dx, n,
                           act);
        return launch_status();
    }
    const unsigned g = map4_grid(n);
    if (!g) return CXM_E_TOO_LARGE;
    switch (act) {
        case CXM_ACT_RELU:
            hipLaunchKernelGGL(k_zip4<ActBwdF<CXM_ACT_RELU>>, dim3(g), dim3(kBlock), 0, hs(s), ActBwdF<CXM_ACT_RELU>{},
                               y, dy, dx, n);
            break;
        case CXM_ACT_SIGMOID:
            hipLaunchKernelGGL(k_zip4<ActBwdF<CXM_ACT_SIGMOID>>, dim3(g), dim3(kBlock), 0, hs(s),
                               ActBwdF<CXM_ACT_SIGMOID>{}, y, dy, dx, n);
            break;
        default:
            hipLaunchKernelGGL(k_zip4<ActBwdF<CXM_ACT_TANH>>, dim3(g), dim3(kBlock), 0, hs(s), ActBwdF<CXM_ACT_TANH>{},
                               y, dy, dx, n);
    }
    return launch_status();
}

int cxm_reduce_sum_bwd_f32(const float *dz, float *dx, size_t outer, size_t dim, size_t inner, int mean,
                           cxm_stream_t s) {
    if (!dz || !dx || (mean != 0 && mean != 1)) return CXM_E_INVALID;
    if (outer == 0 || dim == 0 || inner == 0) return CXM_OK;
    if (outer > SIZE_MAX / dim / inner) return CXM_E_TOO_LARGE;
    return mean ? sum_bwd_t<true>(dz, dx, outer, dim, inner, hs(s)) : sum_bwd_t<false>(dz, dx, outer, dim, inner, hs(s));
}

int cxm_sgd_f32(float *w, const float *g, float lr, size_t n, cxm_stream_t s) {
    if (!w || !g) return CXM_E_INVALID;
    if (n == 0) return CXM_OK;
    if (aligned16(w) && aligned16(g)) {
        const unsigned grid = map4_grid(n);
        if (!grid) return CXM_E_TOO_LARGE;
        hipLaunchKernelGGL(k_zip4<SgdF>, dim3(grid), dim3(kBlock), 0, hs(s), SgdF{lr}, w, g, w, n);
    } else {
        hipLaunchKernelGGL(k_sgd_scalar, dim3(stream_grid((n + 3) / 4)), dim3(kBlock), 0, hs(s), w, g, lr, n);
    }
    return launch_status();
}

}  // extern "C"
