// Stateless fp32-boundary operators: bf_cuda_gemm_f32 and bf_cuda_conv2d_f32
// (drop-ins for reference src/cuda_ops.cu:147-208).
//
// Both multiply on the bf16 matrix cores.  Operands arrive as fp32 and are
// rounded to bf16 while they are staged into LDS; the convolution never
// materialises an im2col matrix (conv_direct.h reads every tap from one staged
// patch; conv_core.h gathers taps straight from NCHW for the shapes that does
// not take).
#include "bf_cuda_ops.h"
#include "conv_core.h"
#include "conv_direct.h"
#include "internal.h"

#include <climits>
#include <cstring>

using namespace bfhip;

namespace {

bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

template <class T, bool VEC>
void gemm_f32_launch(const float *x, const float *w, const float *b, float *y, int M, int K,
                     int N, int relu, hipStream_t s) {
    LoadRowsF32<T::BM, T::BK, T::kThreads, VEC> al{x, K, M, K};
    LoadRowsF32<T::BN, T::BK, T::kThreads, VEC> bl{w, K, N, K};
    EpiRowsF32 epi{y, b, N, M, N, relu};
    launch_gemm<T>(al, bl, epi, M, N, K, s);
}

// Short reductions (K <= 128, the linear 11264 x 96 -> 288):
// one pass per row panel with every load issued up front, instead of the
// tiled core's K/32 rounds of global -> registers -> LDS -> MFMA.  The grid
// is (row panels of 128) x (2 column halves).  A workgroup copies its half
// of W into LDS as fp32 with buffer_load ... lds (no register round trip;
// the 16-byte chunks of each row are XOR-swizzled so that fragment reads are
// conflict-free), while each wave loads its 16 x K slice of X straight into
// MFMA operand registers.  It then walks its column blocks: Y^T block =
// W block * X^T on the bf16 MFMA, W fragments rounded to bf16 as they are
// read, so each lane ends up holding 4 consecutive output columns of one row
// and stores them as one float4.  Operands are rounded to bf16 exactly as the
// tiled core rounds them, the k order of the accumulation is the same
// (32-deep MFMA steps in increasing k) and the bias is added after it, so the
// two paths agree bit for bit.  Requires K % 4 == 0, N % 4 == 0 and 16-byte
// aligned X, W, bias and Y.  Measured on MI355X at M = 11264, K = 96,
// N = 288 (HIP-graph replays): 8.05 us (the tiled core: 8.8 us).
// Staging W per workgroup is what costs: with all 288 columns in one
// workgroup and W converted through registers it took 6.3 of 12.5 us; half
// the columns per workgroup and eight waves brought that form to 7.8 us,
// and the same kernel with no W, X or Y traffic still takes 3.1 us.
constexpr int kPanelWaves = 8;
constexpr int kPanelThreads = kPanelWaves * kWave;
constexpr int kPanelRows = 16 * kPanelWaves;
constexpr int kPanelMaxFrags = 9;  // column blocks per half: N <= 288

inline int panel_cols(int N) { return 16 * (((N + 15) / 16 + 1) / 2); }  // per column half
inline size_t panel_lds_bytes(int N, int ks) { return (size_t)panel_cols(N) * 8 * ks * 16; }

template <int KS>
__global__ __launch_bounds__(kPanelThreads) void gemm_f32_panel_kernel(
    const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
    float *__restrict__ y, int M, int K, int N, int NC, int relu) {
    extern __shared__ __attribute__((aligned(16))) float swf[];
    constexpr int kChunks = 8 * KS;  // 16-byte chunks per padded W row
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = (int)blockIdx.y * NC;
    const int nc = min(NC, N - n0);  // columns of this half
    const int row = (int)blockIdx.x * kPanelRows + 16 * wave + (lane & 15);
    const bool row_ok = row < M;

    // W rows n0 .. n0 + NC - 1 -> LDS: LDS chunk L = n * kChunks + s holds
    // global chunk c = s ^ (n & 7) of row n0 + n (zero past N or K).
    const __amdgpu_buffer_rsrc_t rsrc = buffer_rsrc(w, (uint32_t)N * K * 4);
    const int total = NC * kChunks;
    for (int i = wave; i * 64 < total; i += kPanelWaves) {
        const int L = 64 * i + lane;
        const int n = L / kChunks, c = (L % kChunks) ^ (n & 7);
        const bool in = L < total && n < nc && 4 * c < K;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsrc, (__attribute__((address_space(3))) void *)(swf + 256 * i), 16,
            in ? (uint32_t)(((n0 + n) * K + 4 * c) * 4) : kDmaOutOfRange, 0, 0, 0);
    }
    // This lane's X operands (row `row`, k = 32 ks + 8 (lane >> 4) .. + 7)
    // and the bias of its column quads 16 f + 4 (lane >> 4), f < NC / 16.
    const int col4 = 4 * (lane >> 4);
    float4 xa[KS][2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 32 * ks + 8 * (lane >> 4) + 4 * h;
            xa[ks][h] = row_ok && k < K ? *reinterpret_cast<const float4 *>(x + (size_t)row * K + k)
                                        : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    float4 bq[kPanelMaxFrags];
#pragma unroll
    for (int f = 0; f < kPanelMaxFrags; ++f)
        bq[f] = bias && 16 * f + col4 < nc ? *reinterpret_cast<const float4 *>(bias + n0 + 16 * f + col4)
                                           : make_float4(0.f, 0.f, 0.f, 0.f);
    bf16x8 xb[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const float t[8] = {xa[ks][0].x, xa[ks][0].y, xa[ks][0].z, xa[ks][0].w,
                            xa[ks][1].x, xa[ks][1].y, xa[ks][1].z, xa[ks][1].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) xb[ks][e] = to_bf16(t[e]);
    }
    wait_vmcnt<0>();
    __syncthreads();

    const int nl = lane & 15;  // the lane's W row within a column block
#pragma unroll
    for (int f = 0; f < kPanelMaxFrags; ++f) {
        if (16 * f >= NC) break;
        const int n = 16 * f + nl;
        const float *wr = swf + n * kChunks * 4;
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int c = 8 * ks + 2 * (lane >> 4);
            const float4 lo = *reinterpret_cast<const float4 *>(wr + 4 * (c ^ (n & 7)));
            const float4 hi = *reinterpret_cast<const float4 *>(wr + 4 * ((c + 1) ^ (n & 7)));
            const bf16x8 a = {to_bf16(lo.x), to_bf16(lo.y), to_bf16(lo.z), to_bf16(lo.w),
                              to_bf16(hi.x), to_bf16(hi.y), to_bf16(hi.z), to_bf16(hi.w)};
            acc = mfma16(a, xb[ks], acc);
        }
        // acc[r]: output column n0 + 16 f + 4 (lane >> 4) + r of row `row`.
        const int col = 16 * f + col4;
        float4 v = make_float4(acc[0] + bq[f].x, acc[1] + bq[f].y, acc[2] + bq[f].z, acc[3] + bq[f].w);
        if (relu) {  // NaN passes through, as in the reference's ReLU
            v.x = v.x < 0.f ? 0.f : v.x; v.y = v.y < 0.f ? 0.f : v.y;
            v.z = v.z < 0.f ? 0.f : v.z; v.w = v.w < 0.f ? 0.f : v.w;
        }
        if (row_ok && col < nc) *reinterpret_cast<float4 *>(y + (size_t)row * N + n0 + col) = v;
    }
}

// Whether the panel kernel takes the shape.
bool gemm_f32_panel_takes(const float *x, const float *w, const float *b, const float *y, int K,
                          int N) {
    return K <= 128 && !(K & 3) && !(N & 3) && N > 144 &&
           N <= 2 * 16 * kPanelMaxFrags && (long long)N * K * 4 < (1ll << 31) && aligned16(x) &&
           aligned16(w) && aligned16(y) && (!b || aligned16(b)) &&
           panel_lds_bytes(N, (K + 31) / 32) <= 65536;
}

void gemm_f32_panel(const float *x, const float *w, const float *b, float *y, int M, int K, int N,
                    int relu, hipStream_t s) {
    const int ks = (K + 31) / 32;
    const size_t lds = panel_lds_bytes(N, ks);
    const dim3 grid((M + kPanelRows - 1) / kPanelRows, 2);
    const int nc = panel_cols(N);
    switch (ks) {
        case 1: hipLaunchKernelGGL(gemm_f32_panel_kernel<1>, grid, dim3(kPanelThreads), lds, s, x, w, b, y, M, K, N, nc, relu); break;
        case 2: hipLaunchKernelGGL(gemm_f32_panel_kernel<2>, grid, dim3(kPanelThreads), lds, s, x, w, b, y, M, K, N, nc, relu); break;
        case 3: hipLaunchKernelGGL(gemm_f32_panel_kernel<3>, grid, dim3(kPanelThreads), lds, s, x, w, b, y, M, K, N, nc, relu); break;
        default: hipLaunchKernelGGL(gemm_f32_panel_kernel<4>, grid, dim3(kPanelThreads), lds, s, x, w, b, y, M, K, N, nc, relu); break;
    }
}

// Few or thin outputs: one wave per 16 x 16 output tile, no LDS staging.  The
// lanes load their fp32 operand fragments (lane l: row l & 15, eight k at
// 8 (l >> 4)) kAhead MFMA steps ahead and round them in registers; KW waves
// of a workgroup take consecutive shares of the steps and their partial tiles
// are added in LDS in wave order.  Bound by load latency: a step costs about
// 0.8 us and KW of them run side by side, where the tiled core's k-loop takes
// 1 us per 128 columns.  Every tile reads its own rows of both operands, so
// this loses once the 16 x 16 tiles outnumber the CUs several times.  WM tiles
// below one another share a workgroup when the reduction is short (KW = 1).
// MI355X, eight waves against the best tiled core: 200 x 128 -> 256 2.8 vs 3.0
// us, 1068 x 744 -> 41 4.6 vs 8.0, 7 x 1340 -> 2404 5.5 vs 12, 6 x 2386 -> 4 12
// vs 72; four tiles, one wave each: 100000 x 8 -> 16 4.8 vs 8.1.
template <int WM, int KW, bool VEC>
__global__ __launch_bounds__(64 * WM * KW) void gemm_f32_thin_kernel(
    const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
    float *__restrict__ y, int M, int K, int N, int tiles_n, int relu) {
    constexpr int kAhead = 4;
    static_assert(WM == 1 || KW == 1, "one tile per workgroup when the waves split the reduction");
    __shared__ f32x4 part[KW > 1 ? (KW - 1) * 64 : 1];
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int kw = KW > 1 ? wave : 0, pid = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int m0 = 16 * (pid / tiles_n * WM + (KW > 1 ? 0 : wave)), n0 = pid % tiles_n * 16;
    const int steps = (K + 31) / 32, per = (steps + KW - 1) / KW;
    const int s0 = kw * per, s1 = min(steps, s0 + per);
    const uint32_t row = (uint32_t)K * 4u, at = (uint32_t)(lane & 15) * row;
    // Rows past M or N and columns past K read as zero.
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(x + (size_t)min(m0, M) * K, (uint32_t)max(0, min(16, M - m0)) * row);
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(w + (size_t)n0 * K, (uint32_t)min(16, N - n0) * row);

    float xv[kAhead][8], wv[kAhead][8];
    auto fetch = [&](__amdgpu_buffer_rsrc_t r, uint32_t k, float (&v)[8]) {
        if constexpr (VEC) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 f = buffer_f32x4(r, k + 4 * h < (uint32_t)K ? at + 4u * k + 16 * h : kDmaOutOfRange);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * h + e] = f[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = buffer_f32(r, k + e < (uint32_t)K ? at + 4u * (k + e) : kDmaOutOfRange);
        }
    };
    auto load = [&](int p, int s) {
        const uint32_t k = 32u * s + 8u * (lane >> 4);
        fetch(xr, k, xv[p]);
        fetch(wr, k, wv[p]);
    };
#pragma unroll
    for (int p = 0; p < kAhead; ++p)
        if (s0 + p < s1) load(p, s0 + p);
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += kAhead) {
#pragma unroll
        for (int p = 0; p < kAhead; ++p) {
            if (s + p >= s1) break;
            bf16x8 a, b;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                a[e] = to_bf16(wv[p][e]);
                b[e] = to_bf16(xv[p][e]);
            }
            if (s + p + kAhead < s1) load(p, s + p + kAhead);
            acc = mfma16(a, b, acc);
        }
    }
    if constexpr (KW > 1) {
        if (kw > 0) part[(kw - 1) * 64 + lane] = acc;
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int q = 0; q < KW - 1; ++q) acc += part[q * 64 + lane];
    }
    // acc[r]: column n0 + 4 (lane >> 4) + r of row m0 + (lane & 15).
    const int col = n0 + 4 * (lane >> 4), r = m0 + (lane & 15);
    if (col >= N || r >= M) return;
    const float4 bq = load_quad(bias, col, N);
    const float bv[4] = {bq.x, bq.y, bq.z, bq.w};
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = acc[e] + bv[e];
        if (relu && v[e] < 0.f) v[e] = 0.f;  // NaN passes through
    }
    float *o = y + (size_t)r * N + col;
    if (col + 3 < N && ((uintptr_t)o & 15) == 0) {
        *reinterpret_cast<float4 *>(o) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col + e < N) o[e] = v[e];
    }
}

template <int WM, int KW, bool VEC>
void gemm_f32_thin_launch(const float *x, const float *w, const float *b, float *y, int M, int K,
                          int N, int relu, hipStream_t s) {
    const int tiles_n = (N + 15) / 16, tiles_m = (M + 16 * WM - 1) / (16 * WM);
    hipLaunchKernelGGL((gemm_f32_thin_kernel<WM, KW, VEC>), dim3(tiles_m * tiles_n), dim3(64 * WM * KW),
                       0, s, x, w, b, y, M, K, N, tiles_n, relu);
}

enum GemmRoute {
    kGemmNone = -1, kGemm128, kGemm64, kGemm32, kGemmThinSplit, kGemmThinRows, kGemmWide, kGemmPanel, kGemm128x32, kGemm128x64
};
using Gemm128 = Tile<128, 128, 64, 2, 4>;
using Gemm64 = Tile<64, 64, 64, 2, 2>;
using Gemm32 = Tile<32, 32, 128, 2, 2>;
using Gemm128x32 = Tile<128, 32, 32, 4, 1>;
using Gemm128x64 = Tile<128, 64, 32, 4, 1>;
using GemmWide = Tile<128, 128, 32, 2, 2>;

// What a launch takes, in microseconds: launch + sqrt(fetch^2 + wait^2) + store
// per megabyte of Y, with
//   fetch: rounds of one workgroup per CU, each its operands' KB / rate + each,
//          but no less than all workgroups' KB at `flow` per CU;
//   wait:  rounds of per_cu workgroups per CU, each its k-blocks x block.
struct GemmCost {
    GemmRoute route;
    int rows, cols, depth, per_cu, threads;  // the workgroup's tile and its k-block
    float launch, each, rate, block, store, flow;
};
// Fitted on MI355X to the times of every kernel at 3989 shapes (rows to
// 400 000, K and N to 8192, most of them spread over the logarithm of sizes up
// to 2.5 G products; a third with K <= 128), apart for operands that are loaded
// as floats (first) and as float4.
constexpr GemmCost kGemmCosts[2][7] = {
    {{kGemm128, 128, 128, 64, 2, Gemm128::kThreads, 2.68f, 1.28f, 20.5f, 2.37f, 0.419f, 19.6f},
     {kGemm64, 64, 64, 64, 4, Gemm64::kThreads, 2.56f, 0.521f, 19.4f, 1.57f, 0.369f, 18.6f},
     {kGemm32, 32, 32, 128, 4, Gemm32::kThreads, 2.35f, 0.336f, 9.5f, 1.5f, 0.361f, 8.82f},
     {kGemmThinSplit, 16, 16, 256, 4, 8 * kWave, 2.21f, 0.165f, 16.9f, 1.03f, 1.44f, 13.f},
     {kGemmThinRows, 64, 16, 32, 8, 4 * kWave, 2.41f, 0.283f, 64.2f, 0.801f, 0.393f, 9.44f},
     {kGemm128x32, 128, 32, 32, 4, Gemm128x32::kThreads, 2.64f, 0.f, 15.6f, 1.21f, 0.447f, 80.f},
     {kGemm128x64, 128, 64, 32, 4, Gemm128x64::kThreads, 2.73f, 0.f, 17.4f, 1.45f, 0.432f, 21.6f}},
    {{kGemm128, 128, 128, 64, 2, Gemm128::kThreads, 3.67f, 0.502f, 85.5f, 1.05f, 0.229f, 60.6f},
     {kGemm64, 64, 64, 64, 4, Gemm64::kThreads, 2.87f, 0.473f, 158.f, 0.924f, 0.192f, 70.9f},
     {kGemm32, 32, 32, 128, 4, Gemm32::kThreads, 2.64f, 0.398f, 1000.f, 0.881f, 0.253f, 77.1f},
     {kGemmThinSplit, 16, 16, 256, 4, 8 * kWave, 2.32f, 0.326f, 125.f, 0.453f, 0.71f, 40.8f},
     {kGemmThinRows, 64, 16, 32, 8, 4 * kWave, 2.66f, 0.183f, 1000.f, 0.264f, 0.306f, 35.2f},
     {kGemm128x32, 128, 32, 32, 4, Gemm128x32::kThreads, 2.9f, 0.348f, 1000.f, 0.679f, 0.225f, 65.1f},
     {kGemm128x64, 128, 64, 32, 4, Gemm128x64::kThreads, 3.f, 0.522f, 173.f, 0.781f, 0.215f, 69.1f}}};
constexpr GemmCost kPanelCost = {kGemmPanel, kPanelRows, 0, 32, 2, kPanelThreads, 2.89f, 0.f, 55.1f, 0.0696f, 0.202f, 10000.f};

// The kernel with the least estimated time of those whose grid a launch holds.
// At those shapes the choice costs 0.9 % over the fastest kernel in the mean. At
// 14 of them it is more than 4 % slower than the tile that N alone used to name
// (128 x 32 to N = 32, 128 x 64 to 64, the panels or 32 x 144 from 145 to 288,
// four waves on 128 x 128 elsewhere): at most 12 % up to 2.5 G products, 36 % for
// 10 882 x 129 -> 3104.  With estimates that left out the stores and took one set
// of rates for both load widths, and the panels only from 10 240 rows on, it
// cost 4.8 %: 17 406 x 14 -> 13 6.3 us (now 3.9; the tile by N 4.6), 9000 x 8 ->
// 200 7.7 (panels: 4.5), 2865 x 337 -> 277 41 (17; 26).  Others: 4224 x 384 ->
// 1536 33.1 -> 18.8 us (265 TFLOP/s; 128 x 128, 64-deep, eight waves), 300 x 1024
// -> 1024 11.1 (32 x 32; 18 with 64 x 64), 35 x 2590 -> 265 402 -> 27.  From some
// 10^9 rows on only four-wave tiles of 128 rows have few enough threads;
// kGemmNone: no kernel has.
template <bool VEC>
GemmRoute gemm_route(int M, int K, int N, bool panel) {
    const auto ceil_div = [](long long a, long long b) { return (a + b - 1) / b; };
    const float mb = (float)M * (float)N * 4e-6f;
    float best = INFINITY;
    GemmRoute pick = kGemmNone;
    // Every call pays for this (35 ns): a kernel whose launch, stores and longer
    // part alone are above the best one needs no square root.
    const auto offer = [&](const GemmCost &c, long long grid, float blocks, float kb) {
        const float rest = best - (c.launch + c.store * mb);
        const float alone = (float)((grid + 255) / 256) * (kb * (1.f / c.rate) + c.each);
        const float all = (float)grid * kb * (1.f / (256.f * c.flow));
        const float fetch = alone > all ? alone : all;
        const float wait = (float)((grid + 256 * c.per_cu - 1) / (256 * c.per_cu)) * blocks * c.block;
        if (fetch >= rest || wait >= rest || !launch_fits(grid, c.threads)) return;
        const float us = c.launch + c.store * mb + sqrtf(fetch * fetch + wait * wait);
        if (us < best) {
            best = us;
            pick = c.route;
        }
    };
#pragma clang loop unroll(full)
    for (int i = 0; i < 7; ++i) {
        const GemmCost &c = kGemmCosts[VEC][i];
        // The thin kernel's fragment offsets are 32-bit; past N = 32 the 128 x 64
        // tile reads X half as often.
        if ((c.route == kGemmThinSplit || c.route == kGemmThinRows) && K > 1 << 20) continue;
        if (c.route == kGemm128x32 && N > 32) continue;
        offer(c, ceil_div(M, c.rows) * ceil_div(N, c.cols), (float)ceil_div(K, c.depth),
              (float)(c.rows + c.cols) * (float)K * 0.004f);
    }
    if (panel) {
        const int cols = panel_cols(N);
        offer(kPanelCost, 2 * ceil_div(M, kPanelRows), (float)(ceil_div(K, 32) * (cols / 16)),
              (float)(kPanelRows + cols) * (float)K * 0.004f);
    }
    if (pick == kGemmNone && launch_fits(ceil_div(M, 128) * ceil_div(N, 128), GemmWide::kThreads)) pick = kGemmWide;
    return pick;
}

template <bool VEC>
void gemm_f32_dispatch(GemmRoute route, const float *x, const float *w, const float *b, float *y,
                       int M, int K, int N, int relu, hipStream_t s) {
    switch (route) {
        case kGemm128: gemm_f32_launch<Gemm128, VEC>(x, w, b, y, M, K, N, relu, s); break;
        case kGemm64: gemm_f32_launch<Gemm64, VEC>(x, w, b, y, M, K, N, relu, s); break;
        case kGemm32: gemm_f32_launch<Gemm32, VEC>(x, w, b, y, M, K, N, relu, s); break;
        case kGemmThinSplit: gemm_f32_thin_launch<1, 8, VEC>(x, w, b, y, M, K, N, relu, s); break;
        case kGemmThinRows: gemm_f32_thin_launch<4, 1, VEC>(x, w, b, y, M, K, N, relu, s); break;
        case kGemm128x32: gemm_f32_launch<Gemm128x32, VEC>(x, w, b, y, M, K, N, relu, s); break;
        case kGemm128x64: gemm_f32_launch<Gemm128x64, VEC>(x, w, b, y, M, K, N, relu, s); break;
        default: gemm_f32_launch<GemmWide, VEC>(x, w, b, y, M, K, N, relu, s); break;
    }
}

bool gemm_f32_vec(const float *x, const float *w, int K) { return (K & 3) == 0 && aligned16(x) && aligned16(w); }

GemmRoute gemm_f32_route(const float *x, const float *w, const float *b, const float *y, int M,
                         int K, int N) {
    if (!gemm_f32_vec(x, w, K)) return gemm_route<false>(M, K, N, false);
    return gemm_route<true>(M, K, N, gemm_f32_panel_takes(x, w, b, y, K, N));
}

template <class T>
void conv_dispatch_tile(const ConvGeom &g, int Co, const float *x, const float *w,
                        const float *b, float *y, int relu, hipStream_t s) {
    LoadConvA<T::BM, T::BK, T::kThreads, 0, 0, SrcNCHW> al{};
    al.src = SrcNCHW{x, g.Ci, g.IH, g.IW};
    al.g = g;
    EpiNCHW epi{y, b, g.M, Co, g.OH * g.OW, relu};
    if (g.transpose) {
        LoadWeightIOHW<T::BN, T::BK, T::kThreads> bl{w, Co, g.K, g.KH * g.KW};
        launch_gemm<T>(al, bl, epi, g.M, Co, g.K, s);
    } else if ((g.K & 3) == 0 && aligned16(w)) {
        LoadRowsF32<T::BN, T::BK, T::kThreads, true> bl{w, g.K, Co, g.K};
        launch_gemm<T>(al, bl, epi, g.M, Co, g.K, s);
    } else {
        LoadRowsF32<T::BN, T::BK, T::kThreads, false> bl{w, g.K, Co, g.K};
        launch_gemm<T>(al, bl, epi, g.M, Co, g.K, s);
    }
}

template <class T>
void conv_direct_launch(const DirectConv &d, int batches, bool vec, bool flat, hipStream_t s) {
    const dim3 grid(d.tiles_y * d.tiles_x * d.tiles_c * batches), block(T::kThreads);
    if (d.up_h) {
        if (vec && flat)
            hipLaunchKernelGGL((conv_direct_kernel<T, true, true, true>), grid, block, 0, s, d);
        else if (vec)
            hipLaunchKernelGGL((conv_direct_kernel<T, true, true, false>), grid, block, 0, s, d);
        else if constexpr (T::BC < 128)  // (the largest tile is not offered to scalar transposed layers)
            hipLaunchKernelGGL((conv_direct_kernel<T, true, false, false>), grid, block, 0, s, d);
    } else if (vec && flat) {
        hipLaunchKernelGGL((conv_direct_kernel<T, false, true, true>), grid, block, 0, s, d);
    } else if (vec) {
        hipLaunchKernelGGL((conv_direct_kernel<T, false, true, false>), grid, block, 0, s, d);
    } else {
        hipLaunchKernelGGL((conv_direct_kernel<T, false, false, false>), grid, block, 0, s, d);
    }
}

// The kernel a convolution runs: a tile of the direct kernel, or the gather core.
enum ConvRoute { kConvBig, kConvMid, kConvLow, kConvMin, kConvGather };
using ConvBig = DirectTile<128, 160, 2, 2, 8, 9, 1>;
using ConvMid = DirectTile<64, 128, 2, 2, 4, 9, 1>;
using ConvLow = DirectTile<32, 64, 1, 4, 4, 9, 1>;
using ConvMin = DirectTile<32, 32, 2, 2, 4, 9, 1>;
struct ConvChoice { ConvRoute route; bool vec, flat; };

// Costs fitted on MI355X to the times of every tile and of the gather core at
// 3799 layers (draws of up to 20 GFLOP, two fifths of them with at most 64
// channels, an eighth with up to 2000 small images), in the terms of DirectCost;
// store: per megabyte of output, of plain and of transposed layers.
struct ConvCost {
    float launch, ends, rate, block, store, store_up;
    float base(float mb, bool up) const { return launch + (up ? store_up : store) * mb; }
};
constexpr ConvCost kDirectCosts[2][4] = {  // single floats, float4
    {{3.33f, 3.8f, 41.7f, 0.f, 0.678f, 1.5f},
     {3.82f, 2.53f, 31.2f, 0.f, 0.358f, 0.624f},
     {3.06f, 1.61f, 42.4f, 0.901f, 0.285f, 0.0485f},
     {3.05f, 1.41f, 40.5f, 0.829f, 0.454f, 0.f}},
    {{4.35f, 3.15f, 46.6f, 0.f, 0.667f, 0.644f},
     {4.99f, 1.68f, 41.1f, 0.f, 0.422f, 0.379f},
     {3.27f, 1.38f, 48.1f, 0.775f, 0.603f, 0.143f},
     {3.16f, 1.31f, 46.7f, 0.624f, 1.f, 0.f}}};
// The gather core with 32, 64 and 128 output channels per tile: ends and rate
// of a tile's operands as fp32, block per 32-deep k-step (times store_up where
// transposed).
constexpr ConvCost kGatherCosts[3] = {
    {4.31f, 0.651f, 8.87f, 2.78f, 0.155f, 2.22f},
    {5.89f, 1.43f, 11.1f, 2.62f, 0.0767f, 3.03f},
    {13.4f, 0.f, 13.5f, 3.42f, 0.251f, 2.4f}};

float conv_gather_estimate(const ConvGeom &g, int Co, float mb) {
    const int id = Co <= 32 ? 0 : Co <= 64 ? 1 : 2, cols = 32 << id, per_cu = id < 2 ? 4 : 2;
    const ConvCost &c = kGatherCosts[id];
    const long long grid = ((long long)g.M + 127) / 128 * ((Co + cols - 1) / cols);
    const float kb = (float)(128 + cols) * (float)g.K * 0.004f, steps = (float)((g.K + 31) / 32);
    const float fetch = (float)((grid + 255) / 256) * (kb / c.rate + c.ends);
    const float wait = (float)((grid + 256 * per_cu - 1) / (256 * per_cu)) * steps * c.block * (g.transpose ? c.store_up : 1.f);
    return c.launch + sqrtf(fetch * fetch + wait * wait) + c.store * mb;
}

// A layer's kernel and, for the direct ones, its plan.
struct ConvPlanned {
    ConvChoice choice;
    DirectPlan plan;
    int tiles_c;
};

// The plan with the least estimate below the gather core's, `limit`; the gather
// core when there is none.  Tiles are planned in the order of their bounds, and
// only while a bound is below the best plan (host time with every tile planned
// in full, and so: 3x3 256 -> 256 on 6 x 32 x 88 2.6 and 0.4 us; 3x3 64 -> 64 on
// 20 x 20 2.4 and 0.25).
ConvPlanned conv_plan(const DirectConv &d, int batches, int kh, bool wv, bool flat, float mb, float limit) {
    struct Offer { float bound; int id; } offers[8];  // id: route + 4 vec
    int count = 0;
    const auto cost = [&](int id) {
        const ConvCost &c = kDirectCosts[id / 4][id % 4];
        return DirectCost{c.base(mb, d.up_h), c.ends, c.rate, c.block};
    };
    const auto with_tile = [](int route, auto f) {
        switch (route) {
            case kConvBig: return f(ConvBig{});
            case kConvMid: return f(ConvMid{});
            case kConvLow: return f(ConvLow{});
            default: return f(ConvMin{});
        }
    };
    for (int id = 0; id < (wv ? 8 : 4); ++id) {
        if (id == kConvBig && d.up_h) continue;  // (no scalar transposed instance)
        const float bound = with_tile(id % 4, [&](auto t) { return direct_bound<decltype(t)>(d, batches, cost(id)); });
        if (bound >= limit) continue;
        int at = count++;
        for (; at > 0 && offers[at - 1].bound > bound; --at) offers[at] = offers[at - 1];
        offers[at] = Offer{bound, id};
    }
    ConvPlanned best{{kConvGather, false, false}, {}, 0};
    for (int i = 0; i < count && offers[i].bound < limit; ++i) {
        const int id = offers[i].id;
        const bool vec = id >= 4;
        with_tile(id % 4, [&](auto t) {
            using T = decltype(t);
            const DirectPlan p = direct_plan<T>(d, batches, kh, vec && !d.up_h, vec && flat, cost(id), limit);
            if (p.us < 0.f) return;
            limit = p.us;
            best = ConvPlanned{{(ConvRoute)(id % 4), vec, vec && flat}, p, (d.columns + T::BC - 1) / T::BC};
        });
    }
    return best;
}

// The plans of the layers that a thread called last: a network calls the same
// few over and over.  An entry is found by everything that a plan depends on,
// and holds no address; a layer that is not there is planned (host time of a
// call: 0.05 us with its plan in the table, 0.1 to 0.5 without).
struct ConvPlanTable {
    static constexpr unsigned kEntries = 32;
    struct Key {
        bf_cuda_conv2d_desc desc;
        int loads;  // 1: float4 weights, 2: float4 patch
    };
    struct Entry {
        Key key;  // zero batches: empty
        ConvPlanned planned;
    } entries[kEntries];
    Entry &at(const Key &k) {
        static_assert(sizeof(Key) == 16 * sizeof(int), "compared as words");
        const int *w = reinterpret_cast<const int *>(&k);
        unsigned h = 0;
        for (int i = 0; i < 16; ++i) h = (h + (unsigned)w[i]) * 0x9e3779b1u;
        return entries[h >> 27];
    }
};

ConvGeom conv_geom(const bf_cuda_conv2d_desc &d) {
    ConvGeom g{};
    g.N = d.batches; g.Ci = d.input_channels; g.IH = d.input_height; g.IW = d.input_width;
    g.OH = d.output_height; g.OW = d.output_width; g.KH = d.kernel_height;
    g.KW = d.kernel_width; g.SH = d.stride_height; g.SW = d.stride_width;
    g.PH = d.padding_height; g.PW = d.padding_width; g.transpose = d.transpose;
    g.M = d.batches * d.output_height * d.output_width;
    g.K = d.input_channels * d.kernel_height * d.kernel_width;
    return g;
}

// The direct kernel's plan for this convolution, or the gather core: when that
// is estimated to be faster (few channels on many pixels, where the direct
// kernel fetches and stores octets of channels that are not there; many images
// smaller than a tile), and for shapes the direct kernel does not take: more
// than 36 taps, a transposed layer whose kernel is not its stride (or padded, or
// cropped), an image or weight tensor of 1 GiB or more, a stride so large that
// no patch fits, or a grid that no launch holds.
//
// Tiles: 128 x 160 (eight loader waves) for full grids, 64 x 128 and 32 x 64
// below, 32 x 32 where the grid would leave CUs idle.  Measured on MI355X against
// the im2col gather: 3x3 256 -> 256 on 6 x 32 x 88 433 -> 39 us (515 TFLOP/s),
// transposed 2x2 256 -> 256 on 90 x 90 376 -> 33 us.  By tile: 3x3 512 -> 128 on
// 64 x 64 27 us with 32 x 64 tiles (40 with 64 x 128, 30 with 32 x 32), 3x3 64 ->
// 64 on 2 x 128 x 128 12 us with 64 x 128 (18 with 128 x 160, 19 with 32 x 64).
// At 9293 layers the choice costs 0.8 % over the fastest kernel in the mean, and
// at 148 of them it is more than 4 % slower than the gather core, by up to 60 %
// (5x5 2 -> 6 on 6 x 87 x 272: 29 us, 19).  By one rate and without the stores,
// the gather core left out where the direct kernel takes the shape, it cost 5.8 %
// and was slower than the gather core at 5.4 %: 1x1 8 -> 8 on 5 x 187 x 470 56 us
// (now 23), 3x3 1 -> 2 on 6 x 72 x 370 26 (10).
ConvChoice conv_direct(const bf_cuda_conv2d_desc *c, const ConvGeom &g, const float *x, const float *w,
                       const float *b, float *y, DirectConv &d) {
    constexpr ConvChoice kNone{kConvGather, false, false};
    d.x = x; d.w = w; d.bias = b; d.y = y;
    d.Ci = c->input_channels; d.relu = c->relu;
    d.IH = c->input_height; d.IW = c->input_width;
    const long long hw = (long long)d.IH * d.IW, taps = (long long)c->kernel_height * c->kernel_width;
    const long long columns = c->output_channels * (c->transpose ? taps : 1);
    const long long x_bytes = 4 * hw * d.Ci, w_bytes = 4 * taps * d.Ci * c->output_channels;
    if (taps > 36 || hw >= 1ll << 28 || x_bytes >= 1ll << 30 || w_bytes >= 1ll << 30) return kNone;
    d.columns = (int)columns;
    d.x_bytes = (uint32_t)x_bytes;
    d.w_bytes = (uint32_t)w_bytes;
    int kh = c->kernel_height;
    if (c->transpose) {
        if (c->kernel_height != c->stride_height || c->kernel_width != c->stride_width ||
            c->padding_height || c->padding_width ||
            c->output_height != (long long)d.IH * kh || c->output_width != (long long)d.IW * c->kernel_width)
            return kNone;
        d.up_h = kh; d.up_w = c->kernel_width; d.up_ow = d.IW;
        d.pairs = kh == 2 && d.up_w == 2 && ((uintptr_t)y & 7) == 0;
        d.khw = d.kw = kh = 1;
        d.SH = d.SW = 1;
    } else {
        d.khw = (int)taps; d.kw = c->kernel_width;
        d.SH = c->stride_height; d.SW = c->stride_width;
        d.PH = c->padding_height; d.PW = c->padding_width;
        d.OH = c->output_height; d.OW = c->output_width;
    }
    // One tap at stride one: the image is one row of pixels.
    const bool one = c->transpose || (d.khw == 1 && d.SH == 1 && d.SW == 1 && !d.PH && !d.PW &&
                                      d.OH == d.IH && d.OW == d.IW);
    if (one) {
        d.OH = d.IH = 1;
        d.OW = d.IW = (int)hw;
    }
    const bool wv = aligned16(w) && (c->transpose ? d.columns % 4 == 0 : (long long)d.Ci * d.khw % 4 == 0);
    const bool flat = wv && one && hw % 4 == 0 && aligned16(x);
    static thread_local ConvPlanTable table;
    const ConvPlanTable::Key key{*c, wv + 2 * flat};
    ConvPlanTable::Entry &e = table.at(key);
    if (std::memcmp(&e.key, &key, sizeof key) != 0) {
        const float mb = (float)g.M * (float)c->output_channels * 4e-6f;
        e.planned = conv_plan(d, c->batches, kh, wv, flat, mb, conv_gather_estimate(g, c->output_channels, mb));
        e.key = key;
    }
    const DirectPlan &p = e.planned.plan;
    d.TH = p.TH; d.TW = p.TW; d.O = p.O; d.patch_w = p.patch_w; d.patch = p.patch;
    d.tiles_y = p.tiles_y; d.tiles_x = p.tiles_x; d.tiles_c = e.planned.tiles_c;
    return e.planned.choice;
}

void conv_direct_run(const ConvChoice &c, const DirectConv &d, int batches, hipStream_t s) {
    switch (c.route) {
        case kConvBig: conv_direct_launch<ConvBig>(d, batches, c.vec, c.flat, s); break;
        case kConvMid: conv_direct_launch<ConvMid>(d, batches, c.vec, c.flat, s); break;
        case kConvLow: conv_direct_launch<ConvLow>(d, batches, c.vec, c.flat, s); break;
        default: conv_direct_launch<ConvMin>(d, batches, c.vec, c.flat, s); break;
    }
}

}  // namespace

extern "C" int bf_cuda_conv2d_f32(const bf_cuda_conv2d_desc *d, const float *input,
                                  const float *weight, const float *bias, float *output,
                                  void *stream, char *error, size_t cap) {
    // Contract checks of reference cuda_ops.cu:150-170, in the same order.
    if (!d || !input || !weight || !output || d->batches <= 0 || d->input_channels <= 0 ||
        d->output_channels <= 0 || d->input_height <= 0 || d->input_width <= 0 ||
        d->kernel_height <= 0 || d->kernel_width <= 0 || d->stride_height <= 0 ||
        d->stride_width <= 0 || d->padding_height < 0 || d->padding_width < 0 ||
        d->output_height <= 0 || d->output_width <= 0 ||
        (d->transpose != 0 && d->transpose != 1) || (d->relu != 0 && d->relu != 1))
        return fail(error, cap, "invalid HIP convolution contract");
    const long long batch_rows = (long long)d->batches * d->output_height;
    if (batch_rows > INT_MAX / d->output_width)
        return fail(error, cap, "HIP convolution is too large");
    const long long channel_reduction = (long long)d->input_channels * d->kernel_height;
    if (channel_reduction > INT_MAX / d->kernel_width)
        return fail(error, cap, "HIP convolution reduction is too large");
    if ((d->output_channels + 15LL) / 16 > 65535)
        return fail(error, cap, "HIP convolution has too many output channels");
    const ConvGeom g = conv_geom(*d);
    const int Co = d->output_channels;
    const long long tiles = ((long long)g.M + 127) / 128 * ((Co + 31LL) / 32);
    if (tiles > INT_MAX) return fail(error, cap, "HIP convolution grid is too large");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    DirectConv direct{};
    const ConvChoice choice = conv_direct(d, g, input, weight, bias, output, direct);
    if (choice.route != kConvGather)
        conv_direct_run(choice, direct, d->batches, s);
    else if (Co <= 32)
        conv_dispatch_tile<Tile<128, 32, 32, 4, 1>>(g, Co, input, weight, bias, output, d->relu, s);
    else if (Co <= 64)
        conv_dispatch_tile<Tile<128, 64, 32, 4, 1>>(g, Co, input, weight, bias, output, d->relu, s);
    else
        conv_dispatch_tile<Tile<128, 128, 32, 2, 2>>(g, Co, input, weight, bias, output, d->relu, s);
    return launch_ok(error, cap, "HIP convolution launch");
}

extern "C" int bf_cuda_gemm_f32(const float *input, const float *weight, const float *bias,
                                float *output, int rows, int in_f, int out_f, int relu,
                                void *stream, char *error, size_t cap) {
    // Contract checks of reference cuda_ops.cu:192-196.
    if (!input || !weight || !output || rows <= 0 || in_f <= 0 || out_f <= 0 ||
        (relu != 0 && relu != 1))
        return fail(error, cap, "invalid HIP GEMM contract");
    if ((out_f + 15LL) / 16 > 65535)
        return fail(error, cap, "HIP GEMM has too many output features");
    if (((long long)rows + 127) / 128 * ((out_f + 31LL) / 32) > INT_MAX)
        return fail(error, cap, "HIP GEMM is too large");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const GemmRoute route = gemm_f32_route(input, weight, bias, output, rows, in_f, out_f);
    if (route == kGemmNone) return fail(error, cap, "HIP GEMM is too large");
    if (route == kGemmPanel)  // short reduction: one pass per row panel
        gemm_f32_panel(input, weight, bias, output, rows, in_f, out_f, relu, s);
    else if (gemm_f32_vec(input, weight, in_f))
        gemm_f32_dispatch<true>(route, input, weight, bias, output, rows, in_f, out_f, relu, s);
    else
        gemm_f32_dispatch<false>(route, input, weight, bias, output, rows, in_f, out_f, relu, s);
    return launch_ok(error, cap, "HIP GEMM launch");
}

extern "C" int bfhip_gemm_route(const float *x, const float *w, const float *b, const float *y,
                                int rows, int in_f, int out_f) {
    return gemm_f32_route(x, w, b, y, rows, in_f, out_f);
}

extern "C" int bfhip_conv_route(const bf_cuda_conv2d_desc *desc, const float *x, const float *w,
                                const float *y, unsigned long long *threads) {
    DirectConv d{};
    const ConvChoice c = conv_direct(desc, conv_geom(*desc), x, w, nullptr, const_cast<float *>(y), d);
    constexpr int kThreads[] = {ConvBig::kThreads, ConvMid::kThreads, ConvLow::kThreads, ConvMin::kThreads};
    *threads = c.route == kConvGather ? 0ull
                                      : (unsigned long long)d.tiles_y * d.tiles_x * d.tiles_c * desc->batches * kThreads[c.route];
    return c.route + 8 * c.vec + 16 * c.flat;
}
