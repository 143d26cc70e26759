// bf16 / fp16 products whose operands go straight from memory to the MFMA's
// registers: small ones, ragged ones, and long-K ones with few tiles.
//
// The 16-bit form of gemm_direct.hip: a workgroup's NW waves compute one
// 32 WI x 32 WJ tile, wave w over the 16-k blocks w, w + NW, ..., and meet in
// LDS in wave order; K is split over workgroups as well when there are too
// few tiles.  The staged kernels of gemm16.hip run 256x2077x256 (A^T B) as
// four workgroups, and read an operand whose rows are no multiple of 8
// element by element.
//
// Operands.  v_mfma_f32_32x32x16 takes eight consecutive k per lane, k = 8 lhi
// + 0..7 of a 16-k block.  An operand whose k runs along its rows gives them
// with one 128-bit load per 32 rows (2-byte aligned: unaligned global loads
// are on); one stored [K, M] or [K, N] gives W adjacent columns of one k per
// lane (columns W l32 ..), eight loads whose halves are paired up with
// v_perm.  Rows and columns past the end re-read the last ones; their products
// are not stored.
#include "gemm16.hpp"
#include "gemm_epi.hpp"

namespace cxm {
namespace {

typedef unsigned u32x4u __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned u32u __attribute__((aligned(2)));
typedef unsigned u32x2u __attribute__((ext_vector_type(2), aligned(2)));

constexpr int kDepth = 3;  // 16-k blocks in flight per wave

// k-contiguous operand X[r][k] or not: X[k][r]; W blocks of 32 rows.
template <bool KC, int W>
struct Side16 {
    const uint16_t *base;  // uniform: the tile's first row (KC) or column
    size_t ld;
    unsigned off[KC ? W : 1];  // bytes from base to this lane's data of k block 0
    unsigned sel;              // !KC, W = 2: v_perm selector of block 0 (the high halves where the pair was moved back)
    static constexpr int kRaw = KC ? 4 * W : 8;

    __device__ __forceinline__ void init(const uint16_t *X, size_t r0, size_t rows, size_t ldx, int l32, int lhi) {
        ld = ldx;
        sel = 0x05040100u;
        if constexpr (KC) {
            base = X + r0 * ldx;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const size_t r = r0 + 32 * i + l32;
                off[i] = static_cast<unsigned>((((r < rows ? r : rows - 1) - r0) * ldx + 8 * lhi) * sizeof(uint16_t));
            }
        } else {
            const size_t c = r0 + W * l32, last = rows - W;
            const size_t cc = c < last ? c : last;
            if (c == cc + 1) sel = 0x07060302u;
            const size_t back = r0 < last ? 0 : r0 - last;  // a last tile of one column
            base = X + r0 - back;
            off[0] = static_cast<unsigned>((cc - (r0 - back) + 8 * static_cast<size_t>(lhi) * ldx) * sizeof(uint16_t));
        }
    }
    __device__ __forceinline__ void load(size_t k, unsigned (&f)[kRaw]) const {
        if constexpr (KC) {
            const char *b = reinterpret_cast<const char *>(base + k);
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const u32x4u v = *reinterpret_cast<const u32x4u *>(b + off[i]);
                f[4 * i] = v.x; f[4 * i + 1] = v.y; f[4 * i + 2] = v.z; f[4 * i + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const char *b = reinterpret_cast<const char *>(base + (k + e) * ld) + off[0];
                if constexpr (W == 2) f[e] = *reinterpret_cast<const u32u *>(b);
                else f[e] = *reinterpret_cast<const uint16_t *>(b);
            }
        }
    }
    // The MFMA operand of block i.
    __device__ __forceinline__ u32x4 frag(const unsigned (&f)[kRaw], int i) const {
        if constexpr (KC) {
            return u32x4{f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]};
        } else {
            const unsigned s = i == 0 ? sel : 0x07060302u;
            u32x4 v;
#pragma unroll
            for (int p = 0; p < 4; ++p) v[p] = __builtin_amdgcn_perm(f[2 * p + 1], f[2 * p], s);
            return v;
        }
    }
    // The last, partial block: n < 16 valid k; the others are zero on both sides.
    __device__ __forceinline__ u32x4 frag_tail(size_t k, int n, int lhi, int i) const {
        u32x4 v = {0u, 0u, 0u, 0u};
        const long step = KC ? 1 : static_cast<long>(ld);
        const char *b = reinterpret_cast<const char *>(base + (KC ? k : k * ld)) + off[KC ? i : 0];
        const int col = KC ? 0 : (W == 2 && (i == 1 || sel == 0x07060302u)) ? 1 : 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int kk = 8 * lhi + e;
            const int kc = kk < n ? kk : n - 1;
            const unsigned x = reinterpret_cast<const uint16_t *>(b)[(static_cast<long>(kc) - 8 * lhi) * step + col];
            const unsigned y = kk < n ? x : 0u;
            v[e / 2] |= (e & 1) ? y << 16 : y;
        }
        return v;
    }
};

template <int DT, int WI, int WJ, int NW, bool KCA, bool KCB>
__global__ __launch_bounds__(NW * kWave) void k_gemm16_direct(const uint16_t *__restrict__ A,
                                                              const uint16_t *__restrict__ B, uint16_t *__restrict__ C, size_t M, size_t N, size_t K,
                                                            unsigned wgs, unsigned tiles_n, unsigned splits, size_t kper,
                                                              float *__restrict__ part,
                                                              unsigned *__restrict__ counters) {
    constexpr int TM = 32 * WI, TN = 32 * WJ, LP = TN + 4;
    constexpr int NT = NW * kWave, Q = 32 * TN / 4;  // float4s of a 32-row block
    __shared__ __attribute__((aligned(16))) float sums[NW][32 * LP];
    __shared__ int flag;
    const unsigned wg = xcd_remap(blockIdx.x, wgs);
    const unsigned tile = wg / splits, split = wg - tile * splits;
    const size_t m0 = static_cast<size_t>(tile / tiles_n) * TM, n0 = static_cast<size_t>(tile % tiles_n) * TN;
    const size_t kbeg = static_cast<size_t>(split) * kper;
    const size_t kend = kbeg + kper < K ? kbeg + kper : K;
    const int lane = threadIdx.x & (kWave - 1), l32 = lane & 31, lhi = lane >> 5;
    const unsigned w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

    Side16<KCA, WI> a;
    Side16<KCB, WJ> b;
    a.init(A, m0, M, KCA ? K : M, l32, lhi);
    b.init(B, n0, N, KCB ? K : N, l32, lhi);

    f32x16 acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // whole blocks of this wave: w, w + NW, ... < nb
    const unsigned nb = static_cast<unsigned>((kend - kbeg) / 16);
    const unsigned T = nb > w ? (nb - w + NW - 1) / NW : 0;
    const size_t k0 = kbeg + 16 * static_cast<size_t>(w);
    auto at = [&](unsigned t) { return k0 + static_cast<size_t>(t < T ? t : T - 1) * (16 * NW); };
    unsigned fa[kDepth][Side16<KCA, WI>::kRaw], fb[kDepth][Side16<KCB, WJ>::kRaw];
    auto mul = [&](const unsigned (&x)[Side16<KCA, WI>::kRaw], const unsigned (&y)[Side16<KCB, WJ>::kRaw]) {
        u32x4 u[WI], v[WJ];
#pragma unroll
        for (int i = 0; i < WI; ++i) u[i] = a.frag(x, i);
#pragma unroll
        for (int j = 0; j < WJ; ++j) v[j] = b.frag(y, j);
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int j = 0; j < WJ; ++j) acc[i][j] = mfma16<DT>(u[i], v[j], acc[i][j]);
    };
    if (T > 0) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            a.load(at(d), fa[d]);
            b.load(at(d), fb[d]);
        }
        __builtin_amdgcn_sched_barrier(0);
        unsigned t = 0;
        for (; t + kDepth <= T; t += kDepth) {
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                mul(fa[d], fb[d]);
                a.load(at(t + d + kDepth), fa[d]);
                b.load(at(t + d + kDepth), fb[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int d = 0; d < kDepth; ++d)
            if (t + d < T) mul(fa[d], fb[d]);
    }
    const int rest = static_cast<int>((kend - kbeg) % 16);
    if (rest != 0 && w == nb % NW) {
        const size_t kt = kbeg + 16 * static_cast<size_t>(nb);
        u32x4 v[WJ];
#pragma unroll
        for (int j = 0; j < WJ; ++j) v[j] = b.frag_tail(kt, rest, lhi, j);
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const u32x4 u = a.frag_tail(kt, rest, lhi, i);
#pragma unroll
            for (int j = 0; j < WJ; ++j) acc[i][j] = mfma16<DT>(u, v[j], acc[i][j]);
        }
    }

    // the waves' sums meet in LDS, one 32-row block i of the accumulators at a
    // time (a quarter or half of the LDS, so that more workgroups fit a CU)
    constexpr int PT = (Q + NT - 1) / NT;  // float4s per thread and block
    constexpr bool kAll = Q % NT == 0;     // every thread has PT of them
    float4 v[WI][PT];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        if (i > 0) __syncthreads();
#pragma unroll
        for (int j = 0; j < WJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                sums[w][(8 * (r / 4) + 4 * lhi + (r % 4)) * LP + (KCB ? 32 * j + l32 : WJ * l32 + j)] = acc[i][j][r];
        __syncthreads();
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            const int q = threadIdx.x + p * NT;
            if (!kAll && q >= Q) break;
            const int o = (q / (TN / 4)) * LP + (q % (TN / 4)) * 4;
            v[i][p] = *reinterpret_cast<const float4 *>(&sums[0][o]);
#pragma unroll
            for (int s = 1; s < NW; ++s) {
                const float4 u = *reinterpret_cast<const float4 *>(&sums[s][o]);
                v[i][p].x += u.x; v[i][p].y += u.y; v[i][p].z += u.z; v[i][p].w += u.w;
            }
        }
    }
    if (splits > 1) {
        // four planes, one per component, so that a wave's dword stores are contiguous
        constexpr int PL = TM * TN / 4;
        float *my = part + (static_cast<size_t>(tile) * splits + split) * (TM * TN);
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                const int q = threadIdx.x + p * NT;
                if (!kAll && q >= Q) break;
                float *d = my + i * Q + q;
                st_dev(d, v[i][p].x); st_dev(d + PL, v[i][p].y); st_dev(d + 2 * PL, v[i][p].z); st_dev(d + 3 * PL, v[i][p].w);
            }
        if (!last_block_ticket(ctr(counters, tile), splits, &flag)) return;
        const float *tp = part + static_cast<size_t>(tile) * splits * (TM * TN);
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                const int q = threadIdx.x + p * NT;
                if (!kAll && q >= Q) break;
                v[i][p] = sum_splits(tp + i * Q + q, PL, splits, TM * TN);
            }
    }
    // four elements of one row per thread, element by element at the edge
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            const int q = threadIdx.x + p * NT;
            if (!kAll && q >= Q) break;
            const int ml = q / (TN / 4);
            const size_t row = m0 + (KCA ? 32 * i + ml : WI * ml + i), col = n0 + (q % (TN / 4)) * 4;
            if (row >= M || col >= N) continue;
            const uint16_t h[4] = {H<DT>::store(v[i][p].x), H<DT>::store(v[i][p].y), H<DT>::store(v[i][p].z),
                                   H<DT>::store(v[i][p].w)};
            uint16_t *c = C + row * N + col;
            if (col + 4 <= N) {
                *reinterpret_cast<u32x2u *>(c) =
                    u32x2u{h[0] | static_cast<unsigned>(h[1]) << 16, h[2] | static_cast<unsigned>(h[3]) << 16};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < N) c[e] = h[e];
            }
        }
}

template <int DT, int WI, int WJ, int NW>
int launch_direct16(const uint16_t *A, const uint16_t *B, uint16_t *C, size_t M, size_t K, size_t N, bool ta, bool tb,
                    size_t target, cxm_stream_t st) {
    const DirectPlan p = direct_plan(M, N, K, 32 * WI, 32 * WJ, 16 * NW, kDepth, target);
    float *part = nullptr;
    unsigned *counters = nullptr;
    if (p.splits > 1) {
        Workspace ws;
        const int rc = get_workspace(st, p.tiles, p.tiles * p.splits * (32 * WI * 32 * WJ) * sizeof(float), &ws);
        // a capturing stream without scratch: the kernels of gemm16.hip run the
        // shapes that need none of them and refuse the others
        if (rc == CXM_E_CAPTURE) return kDeclined;
        if (rc) return rc;
        part = static_cast<float *>(ws.scratch);
        counters = ws.counters;
    }
    const size_t wgs = p.tiles * p.splits;
    if (wgs > 0x7fffffu) return kDeclined;
    const dim3 grid(static_cast<unsigned>(wgs)), block(NW * kWave);
    const unsigned nw = static_cast<unsigned>(wgs), tn = static_cast<unsigned>(p.tiles_n), sp = static_cast<unsigned>(p.splits);
    hipStream_t s = reinterpret_cast<hipStream_t>(st);
    if (!ta && !tb)
        hipLaunchKernelGGL((k_gemm16_direct<DT, WI, WJ, NW, true, false>), grid, block, 0, s, A, B, C, M, N, K, nw, tn, sp,
                           p.kper, part, counters);
    else if (!ta)
        hipLaunchKernelGGL((k_gemm16_direct<DT, WI, WJ, NW, true, true>), grid, block, 0, s, A, B, C, M, N, K, nw, tn, sp,
                           p.kper, part, counters);
    else
        hipLaunchKernelGGL((k_gemm16_direct<DT, WI, WJ, NW, false, false>), grid, block, 0, s, A, B, C, M, N, K, nw, tn, sp,
                           p.kper, part, counters);
    return launch_status();
}

// Whether the kernels of gemm16.hip are the faster ones for this product
// (measured, us, direct against ring or staged):
//  * the rings from 128 64x64 tiles up (640x1024x640 6.2 / 11.2, 512x4096x1024
//    18.5 / 29.9, but 2048x1024x1024 15.2 / 11.9); with A stored [K, M], which
//    they transpose first, from 600 (1024^3 7.9 / 14.8, 2048x1024x1024 12.2 /
//    17.0, 1536x1024x1536 16.4 / 17.6, 4096x1024x1024 20.8 / 21.5);
//  * where both operands' rows allow 128-bit loads, 256x256 staged tiles on 200
//    CUs and more (4000x1000x4000 123 / 60), and else whichever estimate is
//    the lower: direct 64x64 tiles by their number times K (A B^T, whose operands
//    both come as 32 strided rows per load, by rounds of 256 of them), staged
//    ones by rounds times K (A B 3000x1600x3000 108 / 77, 3000x520x3000 38 / 43,
//    2504x1000x2504 54 / 49; A^T B 3000x1600x3000 94 / 78, 2600x1600x2600 72 /
//    116; A B^T 1456x1600x1684 46 / 28, 900x1600x1700 33 / 28, 900x520x1700
//    10.5 / 13.1);
//  * A B^T of odd K, where the direct loads are only 2-byte aligned, on 380
//    128x128 tiles and more (3001x777x2003 99 / 89; 3000x500x3008 46 / 135).
bool staged_faster(size_t M, size_t K, size_t N, bool ta, bool tb, bool ring, bool vec) {
    const size_t t64 = ((M + 63) / 64) * ((N + 63) / 64), t128 = ((M + 127) / 128) * ((N + 127) / 128),
                 t256 = ((M + 255) / 256) * ((N + 255) / 256);
    if (ring) return t64 > (ta ? 600 : 128);
    if (!vec) return tb && K % 2 != 0 && t128 >= 380;
    if (t256 >= 200 || (tb && t128 >= 180)) return true;
    if (t64 < 180) return false;
    const double k = static_cast<double>(K);
    if (tb) return 3.0 + (t64 + 255) / 256 * (0.6 + 0.0088 * k) > (t64 > 512 ? 1.0 : 1.05) * (7.0 + 0.014 * k);
    const double direct = 3.0 + (ta ? 26e-6 : 29.5e-6) * t64 * k;
    if (t256 >= 128) return direct > 27.0 + 0.0315 * k;
    return !ta && direct > (t128 <= 256 ? 10.0 + 0.0268 * k : 11.5 + 0.038 * k);
}

template <int DT>
int run_direct16(const uint16_t *A, const uint16_t *B, uint16_t *C, size_t M, size_t K, size_t N, bool ta, bool tb,
                 cxm_stream_t st) {
    const size_t t64 = ((M + 63) / 64) * ((N + 63) / 64);
    // the tile (us, 32x32 / 32x64 / 64x64): 333x2000x517 8.9 / 9.2 / 17, 512x512x512
    // 4.4 / 5.6 / 6.1, 640x1024x640 8.6 / 6.2 / 9.9, 300x4000x1024 29 / 19 / 27,
    // 160x1008x4000 14.6 / 12.2 / 10.1, 1000x1000x1000 15.8 / 11.2 / 10.6
    if (t64 < 64 || (t64 < 100 && K < 1024)) return launch_direct16<DT, 1, 1, 4>(A, B, C, M, K, N, ta, tb, 256, st);
    if (t64 < 180) return launch_direct16<DT, 1, 2, 4>(A, B, C, M, K, N, ta, tb, 256, st);
    return launch_direct16<DT, 2, 2, 4>(A, B, C, M, K, N, ta, tb, 1, st);
}

}  // namespace

int gemm16_direct(const uint16_t *A, const uint16_t *B, uint16_t *C, size_t M, size_t K, size_t N, bool ta, bool tb,
                  int dtype, bool ring, bool vec, cxm_stream_t st) {
    // 32-bit byte offsets within a tile; pairs of columns of a [K, M] / [K, N] operand
    constexpr size_t kMaxLd = size_t(1) << 23;
    if ((ta && tb) || M >= kMaxLd || N >= kMaxLd || K >= kMaxLd || (ta && M < 2) || (!tb && N < 2)) return kDeclined;
    if (staged_faster(M, K, N, ta, tb, ring, vec)) return kDeclined;
    if (dtype == CXM_DT_BF16) return run_direct16<CXM_DT_BF16>(A, B, C, M, K, N, ta, tb, st);
    return run_direct16<CXM_DT_F16>(A, B, C, M, K, N, ta, tb, st);
}

}  // namespace cxm
