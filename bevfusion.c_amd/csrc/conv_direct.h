// Direct NCHW fp32 convolution on the bf16 matrix cores, one launch and no
// workspace: the stateless bf_cuda_conv2d_f32.
//
// A workgroup owns BC output channels x BP output pixels (a TH x TW rectangle
// of one image).  The reduction runs over blocks of 8*O input channels: the
// block's input patch (the rectangle's receptive field) and its weights are
// rounded to bf16 once, on their way into LDS, and every kernel tap then reads
// the same patch at a shifted address.  The im2col form this replaces fetched
// and rounded each input element once per tap with its own index arithmetic.
//
// Reduction order.  One MFMA k-slot (8 consecutive k, one 16-byte LDS unit) is
// one tap of eight channels c0 + o + O*e, e = 0..7: channels O apart, so that
// for a fixed e the slots of a block, r = o*KHW + t, are consecutive floats of
// an OIHW weight row and a wave's weight loads are contiguous runs of O*KHW
// floats (eight consecutive channels per slot would make every lane's address
// a stride of KHW floats).  Slots are taken four to an MFMA step; slots past
// O*KHW read zero on both sides, so that an Inf in either operand reaches only
// the sums it belongs to.
//
// Wave roles.  WC x WP compute waves own the accumulators and only read LDS and
// multiply; LW loader waves fetch the next block into registers meanwhile, and
// round it and write it to LDS between two barriers.  With the loads issued by
// the compute waves, the wait for the fetch path to take them added to the MFMA
// time instead of running beside it (3x3 256 -> 256 on 6 x 32 x 88, MI355X: 62
// us; with loader waves 42).  That launch is bound by its loads: each
// workgroup fetches its 1.2 MB of fp32 weights (float4s where the rows allow;
// single floats took 29 of 70 us), then by the fragment reads of its MFMAs.
//
// A transposed convolution whose kernel equals its stride, without padding,
// is the 1x1 convolution to Co*KHW columns (weights [Ci][Co*KHW]) whose column
// (co, dy, dx) of input pixel (y, x) is output pixel (y*KH + dy, x*KW + dx).
#pragma once

#include "gemm_core.h"

#include <cmath>

namespace bfhip {

// What one launch needs of the shape.  Columns: output channels, or
// (channel, dy, dx) of a transposed convolution.
struct DirectConv {
    const float *x, *w, *bias;
    float *y;
    int Ci, IH, IW, OH, OW;       // OH x OW: pixels the GEMM runs over
    int columns, khw, kw;         // taps of the reduction (1 if transposed)
    int SH, SW, PH, PW;
    int TH, TW, O, patch_w, patch;  // rectangle, octets per block, patch width and pixels
    int tiles_y, tiles_x, tiles_c;
    int relu;
    int up_h, up_w, up_ow;        // transposed: kernel (= stride) and input width (OH = 1: flat pixels)
    int pairs;                    // transposed 2x2 onto an 8-byte aligned output
    uint32_t x_bytes, w_bytes;    // one image of x; all of w
};

template <int BC_, int BP_, int WC_, int WP_, int LW_, int KSTEPS_, int XQ_>
struct DirectTile {
    static constexpr int BC = BC_, BP = BP_, WC = WC_, WP = WP_;
    static constexpr int kLoaders = LW_ * kWave, kThreads = WC * WP * kWave + kLoaders;
    static constexpr int kWaveC = BC / WC, kWaveP = BP / WP;
    static constexpr int kFragC = kWaveC / 16, kFragP = kWaveP / 16;
    static constexpr int kSteps = KSTEPS_, kSlots = 4 * KSTEPS_;  // MFMA steps / slots per block
    // Quads (four 16-byte units) of weights and patch per loader thread.
    static constexpr int kWQ = (BC * KSTEPS_ + kLoaders - 1) / kLoaders, kXQ = XQ_;
    static constexpr int kUnits = 4 * kXQ * kLoaders;  // patch units in LDS
    // One spare unit per slot row: the units of consecutive slots of one
    // column (a wave's weight stores) then fall in distinct banks.
    static constexpr int kWRow = BC + 1;
    static_assert(kWaveC % 16 == 0 && kWaveP % 16 == 0, "wave tile must be 16-aligned");
};

__device__ __forceinline__ float buffer_f32(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, voffset, 0, 0));
}
__device__ __forceinline__ f32x4 buffer_f32x4(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, 0, 0));
}

// WV / XV: the weights / patch are fetched four floats at a time.  WV needs
// weight rows of a multiple of four floats on a 16-byte aligned base and whole
// quads of slots (direct) or columns (transposed); XV one-tap layers whose
// pixel rows are so aligned.
template <class T, bool UP, bool WV, bool XV>
__global__ __launch_bounds__(T::kThreads) void conv_direct_kernel(DirectConv d) {
    __shared__ __attribute__((aligned(16))) bf16x8 sW[T::kSlots * T::kWRow];
    __shared__ __attribute__((aligned(16))) bf16x8 sX[T::kUnits + 1];  // last unit: zero
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int hw = d.IH * d.IW, slots = d.O * d.khw, steps = (slots + 3) / 4;
    const int blocks = (d.Ci + 8 * d.O - 1) / (8 * d.O);

    int pid = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int c0 = (pid % d.tiles_c) * T::BC;  // first column
    pid /= d.tiles_c;
    const int x0 = (pid % d.tiles_x) * d.TW;
    pid /= d.tiles_x;
    const int y0 = (pid % d.tiles_y) * d.TH, n = pid / d.tiles_y;

    if (wave >= T::WC * T::WP) {  // loader (wave-uniform branch)
        const int t = tid - T::WC * T::WP * kWave;
        // Units in use; a wave skips the quads past them.
        const int xunits = d.O * d.patch, wunits = T::BC * slots;
        const uint32_t xstep = (uint32_t)d.O * hw * 4u;  // bytes between a unit's channels
        const uint32_t wstep = (uint32_t)d.O * (UP ? d.columns : d.khw) * 4u;

        // Patch: thread t's unit j of quad q is unit 4 (t + q LT) + j (XV) or
        // t + (4 q + j) LT; byte offset of its first channel, out of range
        // for pixels outside the image.
        constexpr int kXN = XV ? T::kXQ : 4 * T::kXQ, kXS = XV ? 4 : 1;
        uint32_t xoff[kXN];
        {
            const int u = kXS * t;
            int o = u / d.patch, p = u - o * d.patch, py = p / d.patch_w, px = p - py * d.patch_w;
            const int so = kXS * T::kLoaders / d.patch, sp = kXS * T::kLoaders - so * d.patch;
            const int sy = sp / d.patch_w, sx = sp - sy * d.patch_w, ph = d.patch / d.patch_w;
#pragma unroll
            for (int i = 0; i < kXN; ++i) {
                const int iy = y0 * d.SH - d.PH + py, ix = x0 * d.SW - d.PW + px;
                const bool in = o < d.O && (unsigned)iy < (unsigned)d.IH && (unsigned)ix < (unsigned)d.IW;
                xoff[i] = in ? (uint32_t)((o * hw + iy * d.IW + ix) * 4) : kDmaOutOfRange;
                px += sx;
                py += sy;
                if (px >= d.patch_w) { px -= d.patch_w; ++py; }
                if (py >= ph) { py -= ph; ++o; }
                o += so;
            }
        }
        // Weights: quad q is four slots (columns if transposed) of one column
        // (slot); without WV its units are separate (column, slot) pairs.
        // Lanes run along the contiguous direction.
        constexpr int kWN = WV ? T::kWQ : 4 * T::kWQ, kWS = WV ? 4 : 1;
        int wunit[kWN];  // LDS unit, -1: none
        {
            const int run = (UP ? T::BC : slots) / kWS, outer = UP ? slots : T::BC;
            int a = t / run, b = t - a * run;
            const int sa = T::kLoaders / run, sb = T::kLoaders - sa * run;
#pragma unroll
            for (int i = 0; i < kWN; ++i) {
                const int c = UP ? kWS * b : a, s = UP ? a : kWS * b;
                const bool live = a < outer;
                // Direct quads: slot 4 b + j is stored as slot j * steps + b.
                wunit[i] = live ? (UP || !WV ? s : b) * T::kWRow + c : -1;
                a += sa;
                b += sb;
                if (b >= run) { b -= run; ++a; }
            }
        }

        // Byte offset of a unit's first weight, out of range past the columns.
        auto weight_at = [&](int unit) {
            const int at = unit / T::kWRow, c = c0 + unit - at * T::kWRow;  // stored slot, column
            const uint32_t k = UP ? at * d.columns + c : c * d.Ci * d.khw + kWS * at;
            return unit >= 0 && c < d.columns ? 4u * k : kDmaOutOfRange;
        };

        float xv[T::kXQ][4][8], wv[T::kWQ][4][8];
        // A block's channels are read through a buffer that starts at the
        // block and ends with the tensor, so channels past the image's last
        // read as zero (a weight row's are zeroed in store()).  The empty asm
        // keeps the offsets of every unit from being hoisted out of the block
        // loop into registers.
        const char *xbase = (const char *)(d.x + (size_t)n * d.Ci * hw);
        auto load = [&](int b) {
            const size_t xat = (size_t)b * 8 * xstep, wat = (size_t)b * 8 * wstep;
            const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(xbase + xat, d.x_bytes - (uint32_t)xat);
            const __amdgpu_buffer_rsrc_t wr = buffer_rsrc((const char *)d.w + wat, d.w_bytes - (uint32_t)wat);
            const int t0 = t & ~63;  // wave-uniform
#pragma unroll
            for (int i = 0; i < kWN; ++i) {
                if (kWS * (t0 + i * T::kLoaders) >= wunits) break;
                int unit = wunit[i];
                asm volatile("" : "+v"(unit));
                uint32_t at = weight_at(unit);
#pragma unroll
                for (int e = 0; e < 8; ++e, at += wstep) {
                    if constexpr (WV) {
                        const f32x4 f = buffer_f32x4(wr, at);
#pragma unroll
                        for (int j = 0; j < 4; ++j) wv[i][j][e] = f[j];
                    } else {
                        wv[i / 4][i % 4][e] = buffer_f32(wr, at);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < kXN; ++i) {
                if (kXS * (t0 + i * T::kLoaders) >= xunits) break;
                uint32_t at = xoff[i];
                asm volatile("" : "+v"(at));
#pragma unroll
                for (int e = 0; e < 8; ++e, at += xstep) {
                    if constexpr (XV) {
                        const f32x4 f = buffer_f32x4(xr, at);
#pragma unroll
                        for (int j = 0; j < 4; ++j) xv[i][j][e] = f[j];
                    } else {
                        xv[i / 4][i % 4][e] = buffer_f32(xr, at);
                    }
                }
            }
        };
        auto pack = [](const float (&f)[8]) {
            bf16x8 v;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = to_bf16(f[e]);
            return v;
        };
        auto store = [&](int b) {
            const int left = d.Ci - 8 * d.O * b;  // channels from this block on
            const int t0 = t & ~63;
            if (!UP && left < 8 * d.O) {  // channels past Ci hold the next row's weights
#pragma unroll
                for (int i = 0; i < 4 * T::kWQ; ++i) {
                    int unit = wunit[WV ? i / 4 : i];
                    asm volatile("" : "+v"(unit));
                    const int at = unit / T::kWRow, o = (WV ? 4 * at + i % 4 : at) / d.khw;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        wv[i / 4][i % 4][e] = o + d.O * e < left ? wv[i / 4][i % 4][e] : 0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < kWN; ++i) {
                if (kWS * (t0 + i * T::kLoaders) >= wunits) break;
                if constexpr (WV) {
                    if (wunit[i] >= 0)
#pragma unroll
                        for (int j = 0; j < 4; ++j) sW[wunit[i] + j * (UP ? 1 : steps * T::kWRow)] = pack(wv[i][j]);
                } else {
                    if (wunit[i] >= 0) sW[wunit[i]] = pack(wv[i / 4][i % 4]);
                }
            }
#pragma unroll
            for (int i = 0; i < kXN; ++i) {
                if (kXS * (t0 + i * T::kLoaders) >= xunits) break;
                if constexpr (XV) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) sX[4 * (t + i * T::kLoaders) + j] = pack(xv[i][j]);
                } else {
                    sX[t + i * T::kLoaders] = pack(xv[i / 4][i % 4]);
                }
            }
        };

        load(0);
        // The unit that padding slots read, and the weight slots no store fills.
        const bf16x8 zero = {};
        if (t == 0) sX[T::kUnits] = zero;
        for (int u = slots * T::kWRow + t; u < 4 * steps * T::kWRow; u += T::kLoaders) sW[u] = zero;
        for (int b = 0; b < blocks; ++b) {
            store(b);
            lds_barrier();
            if (b + 1 == blocks) break;
            load(b + 1);
            lds_barrier();  // the compute waves are done with this block
        }
        return;
    }

    const int wc = wave % T::WC, wp = wave / T::WC;
    // Fragment addresses: the lane's pixels, and per MFMA step the patch
    // offset of its slot (-1: no such slot).
    int pixel[T::kFragP], soff[T::kSteps];
#pragma unroll
    for (int j = 0; j < T::kFragP; ++j) {
        const int m = wp * T::kWaveP + j * 16 + (lane & 15);
        const int ty = m / d.TW, tx = m - ty * d.TW;
        pixel[j] = ty < d.TH ? ty * d.SH * d.patch_w + tx * d.SW : 0;
    }
#pragma unroll
    for (int i = 0; i < T::kSteps; ++i) {
        const int at = 4 * i + (lane >> 4);
        const int s = WV && !UP ? 4 * (at % steps) + at / steps : at;  // slot stored there
        const int o = s / d.khw, t = s - o * d.khw, ky = t / d.kw;
        soff[i] = s < slots ? o * d.patch + ky * d.patch_w + (t - ky * d.kw) : -1;
    }
    const bf16x8 *wrow = sW + (lane >> 4) * T::kWRow + wc * T::kWaveC + (lane & 15);

    f32x4 acc[T::kFragC][T::kFragP];
#pragma unroll
    for (int i = 0; i < T::kFragC; ++i)
#pragma unroll
        for (int j = 0; j < T::kFragP; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int b = 0; b < blocks; ++b) {
        lds_barrier();
#pragma unroll
        for (int i = 0; i < T::kSteps; ++i) {
            if (i >= steps) break;
            bf16x8 a[T::kFragC], p[T::kFragP];
#pragma unroll
            for (int j = 0; j < T::kFragC; ++j) a[j] = wrow[4 * i * T::kWRow + 16 * j];
#pragma unroll
            for (int j = 0; j < T::kFragP; ++j) p[j] = sX[soff[i] >= 0 ? pixel[j] + soff[i] : T::kUnits];
#pragma unroll
            for (int k = 0; k < T::kFragC; ++k)
#pragma unroll
                for (int j = 0; j < T::kFragP; ++j) acc[k][j] = mfma16(a[k], p[j], acc[k][j]);
        }
        if (b + 1 < blocks) lds_barrier();
    }

    // acc[i][j][r]: column c0 + wc*kWaveC + 16 i + 4 (lane >> 4) + r of pixel j.
    const int row_w = UP ? d.up_ow * d.up_w : d.OW;  // output row
    const size_t plane = UP ? (size_t)d.OW * d.up_h * d.up_w : (size_t)d.OH * d.OW;
    const int planes = UP ? d.columns / (d.up_h * d.up_w) : d.columns;
    float *out = d.y + (size_t)n * planes * plane;
#pragma unroll
    for (int j = 0; j < T::kFragP; ++j) {
        const int m = wp * T::kWaveP + j * 16 + (lane & 15);
        const int ty = m / d.TW;
        int oy = y0 + ty, ox = x0 + m - ty * d.TW;
        if (ty >= d.TH || oy >= d.OH || ox >= d.OW) continue;
        if (UP) {
            oy = ox / d.up_ow;
            ox -= oy * d.up_ow;
        }
#pragma unroll
        for (int i = 0; i < T::kFragC; ++i) {
            const int col = c0 + wc * T::kWaveC + 16 * i + 4 * (lane >> 4);
            if (col >= d.columns) continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = UP ? (col + r) / (d.up_h * d.up_w) : col + r;
                v[r] = acc[i][j][r] + (d.bias && col + r < d.columns ? d.bias[c] : 0.0f);
                if (d.relu && v[r] < 0.0f) v[r] = 0.0f;  // NaN passes through
            }
            if (UP && d.pairs) {  // four columns: one channel's 2x2 pixels
                float *p = out + (size_t)(col >> 2) * plane + (size_t)2 * oy * row_w + 2 * ox;
                *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
                *reinterpret_cast<float2 *>(p + row_w) = make_float2(v[2], v[3]);
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (col + r >= d.columns) break;
                if (UP) {
                    const int taps = d.up_h * d.up_w, c = (col + r) / taps, t = col + r - c * taps;
                    const int dy = t / d.up_w, dx = t - dy * d.up_w;
                    out[(size_t)c * plane + (size_t)(oy * d.up_h + dy) * row_w + ox * d.up_w + dx] = v[r];
                } else {
                    out[(size_t)(col + r) * plane + (size_t)oy * d.OW + ox] = v[r];
                }
            }
        }
    }
}

// What a launch of the direct kernel takes, in microseconds: base + sqrt(fetch^2
// + wait^2), base being its launch and its stores, with
//   fetch: rounds of one workgroup per CU, each the fp32 kilobytes that it
//          fetches over all its blocks / rate + ends (first fetch, stores);
//   wait:  rounds of as many workgroups as fit a CU's LDS, each its blocks x
//          block (fetch round trip, two barriers) + ends.
struct DirectCost {
    float base, ends, rate, block;
};
template <class T>
inline float direct_estimate(const DirectCost &c, long long grid, float blocks, float fetch_kb) {
    constexpr size_t kLds = ((size_t)T::kSlots * T::kWRow + T::kUnits + 1) * sizeof(bf16x8);
    constexpr int kPerCu = kLds > 80 * 1024 ? 1 : kLds > 48 * 1024 ? 2 : 4;
    const float fetch = (float)((grid + 255) / 256) * (fetch_kb / c.rate + c.ends);
    const float wait = (float)((grid + 256 * kPerCu - 1) / (256 * kPerCu)) * (c.block * blocks + c.ends);
    return c.base + sqrtf(fetch * fetch + wait * wait);
}

// The rectangle, channel block and tile counts that tile T gives a layer.
struct DirectPlan {
    float us = -1.f;  // estimate, < 0: no plan
    int TH, TW, O, patch_w, patch, tiles_y, tiles_x;
};

// The fewest blocks that tile T's weight slots take the reduction in.
template <class T>
inline float direct_blocks(const DirectConv &d) {
    const int most = T::kSlots / d.khw;
    return (float)(((d.Ci + 7) / 8 + most - 1) / most);
}

// A bound of tile T's estimates: no rectangle does better than whole tiles of
// pixels, no patch and the fewest blocks.
template <class T>
inline float direct_bound(const DirectConv &d, int batches, const DirectCost &c) {
    const long long grid = ((long long)d.OH * d.OW + T::BP - 1) / T::BP * ((d.columns + T::BC - 1) / T::BC) * batches;
    return 0.999f * direct_estimate<T>(c, grid, direct_blocks<T>(d), 0.032f * (float)(T::BC * d.khw) * (float)((d.Ci + 7) / 8));
}

// Tile T's plan with the least estimate below `limit`; none when no rectangle's
// patch fits, an offset could leave 32 bits or the grid is more than a launch
// holds.  quads: whole quads of slots per block (WV); flat: rectangles of whole
// pixel quads (XV).  A rectangle is dropped as soon as its own bound reaches the
// limit.
template <class T>
inline DirectPlan direct_plan(const DirectConv &d, int batches, int kh, bool quads, bool flat, const DirectCost &c,
                              float limit) {
    const int octets = (d.Ci + 7) / 8, o_step = quads ? (d.khw % 4 == 0 ? 1 : d.khw % 2 == 0 ? 2 : 4) : 1;
    const int most = T::kSlots / d.khw < octets ? T::kSlots / d.khw : octets;  // octets per block, before rounding
    const long long wrow = d.up_h ? d.columns : d.khw, hw = (long long)d.IH * d.IW;
    const long long across = (long long)((d.columns + T::BC - 1) / T::BC) * batches;
    const float fewest = direct_blocks<T>(d);
    DirectPlan best;
    constexpr int kHeights[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 32, 64};
#pragma clang loop unroll(full)
    for (int i = 0; i < 13; ++i) {
        const int th = kHeights[i];
        if (th > T::BP || (th > d.OH && th > 1)) break;
        // The rectangle's columns, spread evenly over the tiles of a row.
        const int in_row = (d.OW + T::BP / th - 1) / (T::BP / th);
        int tw = in_row > 1 ? (d.OW + in_row - 1) / in_row : d.OW;
        if (flat) tw = (tw + 3) / 4 * 4;
        const long long pw = (long long)(tw - 1) * d.SW + d.kw, area = pw * ((long long)(th - 1) * d.SH + kh);
        if (tw * th > T::BP || area > T::kUnits) continue;
        const int ty = (d.OH + th - 1) / th, tx = in_row > 1 ? (d.OW + tw - 1) / tw : 1, patch = (int)area;
        const long long grid = (long long)ty * tx * across;
        const float octet_kb = 0.032f * (float)(T::BC * d.khw + patch);
        if (0.999f * direct_estimate<T>(c, grid, fewest, octet_kb * (float)octets) >= limit) continue;
        int o = T::kUnits / patch;  // octets per block: what fits, spread evenly over the blocks
        if (o > most) o = most;
        if (o < 1) continue;
        const int nb = (octets + o - 1) / o;
        o = ((octets + nb - 1) / nb + o_step - 1) / o_step * o_step;
        if (o * d.khw > T::kSlots || o * patch > T::kUnits) o -= o_step;
        if (o < 1 || 32 * o * hw >= 1ll << 30 || 32 * o * wrow >= 1ll << 30) continue;
        if (!launch_fits(grid, T::kThreads)) continue;
        const float blocks = (float)((octets + o - 1) / o);
        const float us = direct_estimate<T>(c, grid, blocks, blocks * (octet_kb * (float)o));
        if (us < limit) {
            limit = us;
            best = DirectPlan{us, th, tw, o, (int)pw, patch, ty, tx};
        }
    }
    return best;
}

}  // namespace bfhip
