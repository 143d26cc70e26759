// fp32 products whose operands go straight from memory to the MFMA's
// registers: small ones, and ragged ones of any size.
//
// The ring kernel of gemm.hip wants 16-byte aligned operands and 128x128
// tiles; a product of a few hundred rows and columns leaves it on a handful
// of CUs, where one tile of K = 784 takes 37 us of one CU's matrix cores.
// Here a workgroup's NW waves all compute the same 32 WI x 32 WJ tile, each
// over its own 8-k blocks (wave w takes blocks w, w + NW, ...: the four
// blocks of a 128-byte line are read by waves of one CU at about the same
// time), with no LDS and no barrier until the end, where the waves' sums
// meet in LDS in wave order.  K is split over workgroups as well when there
// are too few tiles for the chip.  Bound by MFMA issue with one or two waves
// per SIMD (the loads' latency shows) and, for 32x32 tiles, by L1; 4096x300x4095
// reaches 90 TFLOP/s, 40x784x256 4.9 us.
//
// Operands.  In MFMA e of an 8-k block, lanes 0-31 supply k = 4 lhi + e with
// lhi = 0, lanes 32-63 with lhi = 1.  An operand whose k runs along its rows
// (A [M, K], B [N, K]) gives a lane four k with one dword-aligned 128-bit load
// per 32 rows; one stored [K, M] or [K, N] gives 32 W columns of one k with W
// adjacent floats per lane (columns W l32 .. W l32 + W - 1: block i of the
// accumulator holds columns W l + i).  Rows past the end re-read the last
// one, columns past the end re-read the last W: their products land in
// accumulators that are not stored.
#include "gemm_epi.hpp"

namespace cxm {
namespace {

typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// k-contiguous operand X[r][k] or not: X[k][r]; W blocks of 32 rows.
template <bool KC, int W>
struct Side {
    const float *base;  // uniform: the tile's first row (KC) or column
    size_t ld;
    unsigned off[KC ? W : 1];  // bytes from base to this lane's data of k block 0
    int shift;                 // !KC, W = 2: 1 where the lane's pair was moved back by one column

    __device__ __forceinline__ void init(const float *X, size_t r0, size_t rows, size_t ldx, int l32, int lhi) {
        ld = ldx;
        shift = 0;
        if constexpr (KC) {
            base = X + r0 * ldx;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const size_t r = r0 + 32 * i + l32;
                off[i] = static_cast<unsigned>((((r < rows ? r : rows - 1) - r0) * ldx + 4 * lhi) * sizeof(float));
            }
        } else {
            base = X + r0;
            // the last whole W columns when this lane's run past the end
            const size_t c = r0 + W * l32, last = rows - W;
            const size_t cc = c < last ? c : last;
            shift = c == cc + 1 ? 1 : 0;
            // cc may lie before r0 (a tile of one column): base is moved back with it
            const size_t back = r0 < last ? 0 : r0 - last;
            base -= back;
            off[0] = static_cast<unsigned>((cc - (r0 - back) + 4 * static_cast<size_t>(lhi) * ldx) * sizeof(float));
        }
    }
    // This lane's operands of the 8-k block at k: f[i][e], block i, MFMA e.
    __device__ __forceinline__ void load(size_t k, float (&f)[W][4]) const {
        if constexpr (KC) {
            const char *b = reinterpret_cast<const char *>(base + k);
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const f32x4u v = *reinterpret_cast<const f32x4u *>(b + off[i]);
                f[i][0] = v.x; f[i][1] = v.y; f[i][2] = v.z; f[i][3] = v.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const char *b = reinterpret_cast<const char *>(base + (k + e) * ld);
                if constexpr (W == 2) {
                    const f32x2u v = *reinterpret_cast<const f32x2u *>(b + off[0]);
                    f[0][e] = v.x;
                    f[1][e] = v.y;
                } else {
                    f[0][e] = *reinterpret_cast<const float *>(b + off[0]);
                }
            }
        }
    }
    // What load left for the use: the moved pair's first column is its second float.
    __device__ __forceinline__ void settle(float (&f)[W][4]) const {
        if constexpr (!KC && W == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) f[0][e] = shift ? f[1][e] : f[0][e];
        }
    }
    // The last, partial block: n < 8 valid k; the others are zero on both sides.
    __device__ __forceinline__ void load_tail(size_t k, int n, int lhi, float (&f)[W][4]) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int kk = 4 * lhi + e;
            const bool in = kk < n;
            const int kc = in ? kk : n - 1;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                // off holds 4 lhi: step from there to kc
                const long d = KC ? static_cast<long>(kc) - 4 * lhi : (static_cast<long>(kc) - 4 * lhi) * static_cast<long>(ld);
                const char *b = reinterpret_cast<const char *>(base + (KC ? k : k * ld)) + off[KC ? i : 0];
                const float v = reinterpret_cast<const float *>(b)[d + (KC ? 0 : i)];
                f[i][e] = in ? v : 0.0f;
            }
        }
    }
};

constexpr int kDepth = 3;      // 8-k blocks in flight per wave
// Blocks per run of sums (264 k), a multiple of kDepth.  In one chain of all
// its K / (NW splits) terms a wave's rounding error grows with the square
// root of the chain: 333x8191x517, 2048 terms, 8.1e-7 of the result against
// 64 bits, 3.0e-7 in runs.
constexpr unsigned kRun = 33;

template <int WI, int WJ, int NW, bool KCA, bool KCB, bool RUNS>
__global__ __launch_bounds__(NW * kWave) void k_gemm_direct(const float *__restrict__ A, const float *__restrict__ B,
                                                            float *__restrict__ C, size_t M, size_t N, size_t K,
                                                            unsigned wgs, unsigned tiles_n, unsigned splits, size_t kper,
                                                            Epilogue epi, float *__restrict__ part,
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

    Side<KCA, WI> a;
    Side<KCB, WJ> b;
    a.init(A, m0, M, KCA ? K : M, l32, lhi);
    b.init(B, n0, N, KCB ? K : N, l32, lhi);

    floatx16 acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // RUNS: every kRun blocks the sums so far are added to `total` and begin
    // again from zero (see kRun).
    floatx16 total[WI][WJ];
    if constexpr (RUNS) {
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int j = 0; j < WJ; ++j) total[i][j] = acc[i][j];
    }
    auto close_run = [&] {
        if constexpr (RUNS) {
#pragma unroll
            for (int i = 0; i < WI; ++i)
#pragma unroll
                for (int j = 0; j < WJ; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        total[i][j][r] = total[i][j][r] + acc[i][j][r];
                        acc[i][j][r] = 0.0f;
                    }
        }
    };

    // whole blocks of this wave: w, w + NW, ... < nb
    const unsigned nb = static_cast<unsigned>((kend - kbeg) / 8);
    const unsigned T = nb > w ? (nb - w + NW - 1) / NW : 0;
    const size_t k0 = kbeg + 8 * static_cast<size_t>(w);
    auto at = [&](unsigned t) { return k0 + static_cast<size_t>(t < T ? t : T - 1) * (8 * NW); };
    float fa[kDepth][WI][4], fb[kDepth][WJ][4];
    auto mul = [&](float (&x)[WI][4], float (&y)[WJ][4]) {
        a.settle(x);
        b.settle(y);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < WI; ++i)
#pragma unroll
                for (int j = 0; j < WJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][e], y[j][e], acc[i][j], 0, 0, 0);
    };
    if (T > 0) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            a.load(at(d), fa[d]);
            b.load(at(d), fb[d]);
        }
        __builtin_amdgcn_sched_barrier(0);
        unsigned t = 0;
        for (;;) {
            const unsigned stop = RUNS && T - t > kRun ? t + kRun : T;
            for (; t + kDepth <= stop; t += kDepth) {
#pragma unroll
                for (int d = 0; d < kDepth; ++d) {
                    mul(fa[d], fb[d]);
                    a.load(at(t + d + kDepth), fa[d]);
                    b.load(at(t + d + kDepth), fb[d]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (stop == T) break;
            close_run();
        }
#pragma unroll
        for (int d = 0; d < kDepth; ++d)
            if (t + d < T) mul(fa[d], fb[d]);
    }
    const int rest = static_cast<int>((kend - kbeg) % 8);
    if (rest != 0 && w == nb % NW) {
        float x[WI][4], y[WJ][4];
        a.load_tail(kbeg + 8 * static_cast<size_t>(nb), rest, lhi, x);
        b.load_tail(kbeg + 8 * static_cast<size_t>(nb), rest, lhi, y);
        mul(x, y);
    }
    if constexpr (RUNS) {
        close_run();
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int j = 0; j < WJ; ++j) acc[i][j] = total[i][j];
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
    // epilogue: a float4 of one row per thread, element by element at the edge
    const float *pre_src = epi.sgd ? C : epi.gate;
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            const int q = threadIdx.x + p * NT;
            if (!kAll && q >= Q) break;
            const int ml = q / (TN / 4);
            const size_t row = m0 + (KCA ? 32 * i + ml : WI * ml + i), col = n0 + (q % (TN / 4)) * 4;
            if (row >= M || col >= N) continue;
            const size_t o = row * N + col;
            const float u[4] = {v[i][p].x, v[i][p].y, v[i][p].z, v[i][p].w};
            if (col + 4 <= N) {
                float4 pre = make_float4(0.f, 0.f, 0.f, 0.f), bias = make_float4(0.f, 0.f, 0.f, 0.f);
                if (pre_src) pre = ld4_any<false>(pre_src + o);
                if (epi.bias) bias = ld4_any<false>(epi.bias + col);
                *reinterpret_cast<f32x4u *>(C + o) =
                    f32x4u{epi_value(epi, u[0], bias.x, pre.x), epi_value(epi, u[1], bias.y, pre.y),
                           epi_value(epi, u[2], bias.z, pre.z), epi_value(epi, u[3], bias.w, pre.w)};
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (col + c < N)
                        C[o + c] =
                            epi_value(epi, u[c], epi.bias ? epi.bias[col + c] : 0.0f, pre_src ? pre_src[o + c] : 0.0f);
            }
        }
}

template <int WI, int WJ, int NW>
int launch_direct(const float *A, const float *B, float *C, size_t M, size_t K, size_t N, int ta, int tb,
                  const Epilogue &epi, size_t target, cxm_stream_t st) {
    const DirectPlan p = direct_plan(M, N, K, 32 * WI, 32 * WJ, 8 * NW, kDepth, target);
    float *part = nullptr;
    unsigned *counters = nullptr;
    if (p.splits > 1) {
        Workspace ws;
        const int rc = get_workspace(st, p.tiles, p.tiles * p.splits * (32 * WI * 32 * WJ) * sizeof(float), &ws);
        // a capturing stream without scratch: the kernels of gemm.hip run the
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
#define CXM_DIRECT(KCA, KCB, RUNS)                                                                                    \
    hipLaunchKernelGGL((k_gemm_direct<WI, WJ, NW, KCA, KCB, RUNS>), grid, block, 0, s, A, B, C, M, N, K, nw, tn, sp, \
                       p.kper, epi, part, counters)
    constexpr bool kRuns = NW == 4 && WI * WJ <= 2;
    if (kRuns && p.kper > 8 * NW * kRun) {
        if (!ta && !tb) CXM_DIRECT(true, false, kRuns);
        else if (!ta) CXM_DIRECT(true, true, kRuns);
        else CXM_DIRECT(false, false, kRuns);
    } else {
        if (!ta && !tb) CXM_DIRECT(true, false, false);
        else if (!ta) CXM_DIRECT(true, true, false);
        else CXM_DIRECT(false, false, false);
    }
#undef CXM_DIRECT
    return launch_status();
}

// Estimated times, in us, of a product on the kernels of gemm.hip and on the
// direct tiles: rounds of workgroups over the chip, each its own cost plus its
// k range times the cost per k.  gemm_direct takes the smaller one.

// 128x128 tiles, one workgroup per CU and round: 60 ns per k in the ring, 70
// in the register-staged kernels (78 in the four-wave ones of large grids), 80
// with element loads of one operand, 85 (A B^T 95) of both.
double staged_us(size_t M, size_t N, size_t K, int tb, bool ring, int vecs) {
    const size_t tiles = ((M + 127) / 128) * ((N + 127) / 128), cus = device_cus();
    size_t splits = gemm_splits(tiles, K, cus);
    const size_t step = ring ? 128 : 32, kper = ((K + splits - 1) / splits + step - 1) / step * step;
    splits = (K + kper - 1) / kper;
    const size_t rounds = (tiles * splits + cus - 1) / cus;
    const double per_k = ring ? 0.060 : vecs == 0 ? (tb ? 0.095 : 0.085) : vecs == 1 ? 0.080 : tiles * splits >= 1024 ? 0.078 : 0.070;
    return 3.0 + (splits > 1 ? 4.0 + 0.7 * splits : 0.0) + 7.5 * rounds - 1.5 + rounds * per_k * (splits > 1 ? kper : K);
}

// Direct tiles of 32 wi x 32 wj: kPerK per k of one 32x32 block, by tile and
// form (A B, A^T B, A B^T); more where an odd K puts the rows of a k-contiguous
// operand at odd alignments, for A B^T of long K, and for the splits of A^T B
// (short ones above all).  Of the smallest tiles, a second round only partly there
// costs less than a whole one.
double direct_us(size_t M, size_t N, size_t K, int ta, int tb, size_t wi, size_t wj, size_t nw, size_t target) {
    constexpr double kPerK[3][3] = {{0.0066, 0.0062, 0.0070}, {0.0050, 0.0055, 0.0062}, {0.0043, 0.0045, 0.0047}};
    const size_t blocks = wi * wj;
    const DirectPlan p = direct_plan(M, N, K, 32 * wi, 32 * wj, 8 * nw, kDepth, target);
    const double x = static_cast<double>(p.tiles * p.splits) / device_cus(), k = p.splits > 1 ? p.kper : K;
    double e = kPerK[blocks == 4 ? 2 : blocks - 1][tb ? 2 : ta ? 1 : 0], rounds = ceil(x);
    if (!ta && K % 4 != 0 && (tb || blocks == 1)) e *= blocks == 4 && k >= 4096 ? 1.4 : 1.12;
    else if (blocks == 4 && tb && K >= 2048) e *= p.splits > 1 ? 1.2 : 1.15;
    else if (blocks == 4 && ta && p.splits > 1) e *= k < 1200 ? 1.4 : 1.2;
    if (blocks == 1 && !tb && x > 1.0 && x < 2.0) rounds = 1.4 * x - 0.6 < 2.0 ? 1.4 * x - 0.6 : 2.0;
    return 4.0 + rounds * blocks * ((blocks == 4 ? 0.42 : 0.3) + e * k);
}

}  // namespace

// The tile by the product's size.  Measured (us; 32x32 / 32x64 / 64x64 tiles
// with this K split / ring or, ragged, the register-staged kernels):
//   40x784x256        4.9 /  7.2 /  12   /  35.8
//   512x512x512       5.3 /  7.8 /  11   /  25.3
//   333x2000x517     13.4 / 15.7 /  23   /  35.8
//   640x1024x1024    20.3 / 22.5 /  24   /  28.6
//   1000x1000x1000   26.0 / 22.6 /  24.6 /  42.7
//   1536x1024x1024   39.4 / 32.9 /  40.2 /  42.2
//   3000x700x1500    91.8 / 67.3 /  66.5 / 112.7
//   4100x300x4095   150   / 122  / 111   / 173
//   300x4100x4095 TN 131  / 129  / 122   / 175
//   3072x1024x1024   75.7 / 62.1 /  57.4 /  68.2
//   4096x1024x1024   98.6 / 81.2 /  74.9 /  70.1
//   784x4096x1024 TN 102  / 82.5 /  82.9 /  73.9
// Small grids want many small tiles; a 64x64 tile reads half as much per
// flop, which counts once every CU has two; beyond K = 2048 its splits pay.
// 32x64 tiles of more than 1056 k keep their waves' chains within kRun blocks
// by eight waves instead of four (1203x2000x1500 A B 79 us with four, 81 with
// eight, 93 with runs), for A B^T, whose loads eight waves slow down, by runs
// (106 / 115 / 98).
int gemm_direct(const float *A, const float *B, float *C, size_t M, size_t K, size_t N, int ta, int tb,
                const Epilogue &epi, bool ring, int vecs, cxm_stream_t st) {
    // 32-bit byte offsets within a tile; pairs of columns of a [K, M] / [K, N] operand
    constexpr size_t kMaxLd = size_t(1) << 23;
    if ((ta && tb) || M >= kMaxLd || N >= kMaxLd || K >= kMaxLd || (ta && M < 2) || (!tb && N < 2)) return kDeclined;
    const size_t t64 = ((M + 63) / 64) * ((N + 63) / 64);
    const double staged = staged_us(M, N, K, tb, ring, vecs);
    if (t64 < 200) {
        if (direct_us(M, N, K, ta, tb, 1, 1, 4, 256) > staged) return kDeclined;
        return launch_direct<1, 1, 4>(A, B, C, M, K, N, ta, tb, epi, 256, st);
    }
    if (t64 < 600 && K < 2048) {
        if (direct_us(M, N, K, ta, tb, 1, 2, 4, 256) > staged) return kDeclined;
        if (K > 4 * 8 * kRun && !tb) return launch_direct<1, 2, 8>(A, B, C, M, K, N, ta, tb, epi, 256, st);
        return launch_direct<1, 2, 4>(A, B, C, M, K, N, ta, tb, epi, 256, st);
    }
    const size_t target = K < 2048 ? 1 : 768;
    if (direct_us(M, N, K, ta, tb, 2, 2, 4, target) > staged) return kDeclined;
    return launch_direct<2, 2, 4>(A, B, C, M, K, N, ta, tb, epi, target, st);
}

}  // namespace cxm
