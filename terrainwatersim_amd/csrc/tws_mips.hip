// tws_mips.hip -- the terrain mip chain the reference's renderer samples.
//
// After every frame with at least one step, Terrain::PerformSimulationStep
// regenerates the full mip chain of TerrainData (Terrain.cpp:270-276 ->
// Texture2D::GenMipMaps, Texture2D.cpp:64-68, glGenerateMipmap).  The chain
// has floor(log2(max(W,H))) + 1 levels (Texture.cpp:28-44); level l is
// max(1, W>>l) x max(1, H>>l) RGBA32F texels (r = terrain, g = b = the
// constant fill, a = water depth).
//
// Reduction: the bilinear blit Mesa's llvmpipe uses for glGenerateMipmap.
// Each texel of level l+1 samples level l at its own centre,
// u = (i + 0.5) * ws / wd - 0.5, with lerp(a, b, t) = a + t * (b - a), along
// x first, then y, clamped to the edge.  Halving (ws = 2 wd) is t = 0.5
// between texels 2i and 2i+1 and matches llvmpipe bit for bit; other ratios
// use the exact sample position (double, t rounded once to float).
//
// Blocks of three or four levels are made from one read of the planes, or of the
// last level made, in LDS (k_mip_block); the small end of the chain is one work
// group's (k_mip_tail).

#include <hip/hip_runtime.h>

#include <cmath>

#include "tws.h"
#include "tws_grid.hpp"
#include "tws_runtime.hpp"

namespace tws {

namespace {

__host__ __device__ inline void mip_axis(int i, int ws, int wd, int& i0, int& i1, float& t) {
    if (ws == 2 * wd) {
        i0 = 2 * i;
        i1 = 2 * i + 1;
        t = 0.5f;
        return;
    }
    const double u = ((double)i + 0.5) * (double)ws / (double)wd - 0.5;
    double fl = floor(u);
    if (fl < 0.0) fl = 0.0;
    int a = (int)fl;
    if (a > ws - 1) a = ws - 1;
    i0 = a;
    i1 = a + 1 < ws ? a + 1 : ws - 1;
    t = (float)(u - (double)a);
    if (t < 0.0f) t = 0.0f;
}

__device__ __forceinline__ float mip_lerp(float a, float b, float t) { return a + t * (b - a); }

__device__ __forceinline__ float bilerp(float s00, float s01, float s10, float s11, float tx,
                                        float ty) {
    return mip_lerp(mip_lerp(s00, s01, tx), mip_lerp(s10, s11, tx), ty);
}

// Up to kMipLevels levels at once.  A work group owns a block of kMipSide >> 1
// >> ... texels of each, and computes of every level what its texels of the next
// one read too (one or two texels past its own where a side is odd), in LDS; the
// last block of a row or column takes what the halving left over.  Bound by
// launches and latency up to about 1024^2, by the one read of b and d above.
constexpr int kMipLevels = 4;
constexpr int kMipSide = 32;   // side of a block's first level
constexpr int kMipReach = 40;  // what it computes of that level, at most: a last
                               // block owns 32 + 7, an odd side needs 3 + 2 * 18
constexpr int kMipRows = 8;    // wavefronts of a work group, a row of texels each

struct MipAxis {
    int i0, i1;
    float t;
};

struct MipSpan {
    int first, own, end;  // computed: [first, end), written: [first, own)
};

// Texels of a level of `size`, `up` levels above the block's last one, whose
// next level's span is `next`.
__device__ __forceinline__ MipSpan mip_span(int block, bool last, int side, int up, int size,
                                            int next_size, const MipSpan& next, bool have_next) {
    MipSpan r;
    r.first = min((block * side) << up, size);
    r.own = last ? size : min(((block + 1) * side) << up, size);
    r.end = r.own;
    if (have_next && next.end > next.first) {
        int i0, i1;
        float t;
        mip_axis(next.end - 1, size, next_size, i0, i1, t);
        r.end = max(r.end, i1 + 1);
    }
    return r;
}

// Levels 1..levels of a source of ws x hs: the planes b and d of set `parity`
// (PLANES), or a level of the chain.  g = b = `gb` in every texel.
template <bool PLANES>
__global__ void __launch_bounds__(kWave * kMipRows)
k_mip_block(GridDesc g, int parity, float gb, const float4* __restrict__ src, int ws, int hs,
            float4* __restrict__ dst, int levels) {
    __shared__ float2 s_mip[2][kMipReach * kMipReach];  // {r, a}
    // sample positions of a block's columns and rows, every level: worked out
    // once, since a position between texels takes a division in FP64
    __shared__ MipAxis s_axis[2][kMipLevels][kMipReach];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int side = kMipSide >> (levels - 1);
    const bool last_x = blockIdx.x + 1 == gridDim.x, last_y = blockIdx.y + 1 == gridDim.y;
    MipSpan sx[kMipLevels], sy[kMipLevels];
    int w[kMipLevels], h[kMipLevels];
#pragma unroll
    for (int l = 0; l < kMipLevels; ++l) {
        w[l] = max(1, ws >> (l + 1));
        h[l] = max(1, hs >> (l + 1));
        sx[l] = sy[l] = MipSpan{0, 0, 0};
    }
#pragma unroll
    for (int l = kMipLevels - 1; l >= 0; --l) {
        if (l >= levels) continue;
        constexpr int top = kMipLevels - 1;
        const int n = l < top ? l + 1 : top;
        const bool more = l + 1 < levels;
        sx[l] = mip_span(blockIdx.x, last_x, side, levels - 1 - l, w[l], w[n], sx[n], more);
        sy[l] = mip_span(blockIdx.y, last_y, side, levels - 1 - l, h[l], h[n], sy[n], more);
    }
    const float* d = parity ? g.d[1] : g.d[0];
#pragma unroll
    for (int l = 0; l < kMipLevels; ++l) {
        if (l >= levels) break;
        const int sw = l == 0 ? ws : w[l > 0 ? l - 1 : 0], sh = l == 0 ? hs : h[l > 0 ? l - 1 : 0];
        if (wave == 2 * l && sx[l].first + lane < sx[l].end) {
            MipAxis& x = s_axis[0][l][lane];
            mip_axis(sx[l].first + lane, sw, w[l], x.i0, x.i1, x.t);
        }
        if (wave == 2 * l + 1 && sy[l].first + lane < sy[l].end) {
            MipAxis& y = s_axis[1][l][lane];
            mip_axis(sy[l].first + lane, sh, h[l], y.i0, y.i1, y.t);
        }
    }
    static_assert(kMipRows >= 2 * kMipLevels, "a wavefront for each axis of each level");
    __syncthreads();
#pragma unroll
    for (int l = 0; l < kMipLevels; ++l) {
        if (l >= levels) break;
        const int i = sx[l].first + lane;
        if (i < sx[l].end) {
            const MipAxis ax = s_axis[0][l][lane];
            const int x0 = ax.i0, x1 = ax.i1;
            const float tx = ax.t;
            for (int j = sy[l].first + wave; j < sy[l].end; j += kMipRows) {
                const MipAxis ay = s_axis[1][l][j - sy[l].first];
                const int y0 = ay.i0, y1 = ay.i1;
                const float ty = ay.t;
                float2 v;
                if (l == 0 && PLANES) {
                    const int64_t r0 = (int64_t)y0 * g.pitch, r1 = (int64_t)y1 * g.pitch;
                    v.x = bilerp(g.b[r0 + x0], g.b[r0 + x1], g.b[r1 + x0], g.b[r1 + x1], tx, ty);
                    v.y = bilerp(d[r0 + x0], d[r0 + x1], d[r1 + x0], d[r1 + x1], tx, ty);
                } else if (l == 0) {
                    const float4* r0 = src + (int64_t)y0 * ws;
                    const float4* r1 = src + (int64_t)y1 * ws;
                    const float4 s00 = r0[x0], s01 = r0[x1], s10 = r1[x0], s11 = r1[x1];
                    v.x = bilerp(s00.x, s01.x, s10.x, s11.x, tx, ty);
                    v.y = bilerp(s00.w, s01.w, s10.w, s11.w, tx, ty);
                } else {
                    const MipSpan &px = sx[l > 0 ? l - 1 : 0], &py = sy[l > 0 ? l - 1 : 0];
                    const float2* up = s_mip[(l & 1) ^ 1];
                    const float2* r0 = up + (y0 - py.first) * kMipReach - px.first;
                    const float2* r1 = up + (y1 - py.first) * kMipReach - px.first;
                    const float2 s00 = r0[x0], s01 = r0[x1], s10 = r1[x0], s11 = r1[x1];
                    v.x = bilerp(s00.x, s01.x, s10.x, s11.x, tx, ty);
                    v.y = bilerp(s00.y, s01.y, s10.y, s11.y, tx, ty);
                }
                s_mip[l & 1][(j - sy[l].first) * kMipReach + lane] = v;
                if (i < sx[l].own && j < sy[l].own) {
                    const float c = bilerp(gb, gb, gb, gb, tx, ty);
                    dst[(int64_t)j * w[l] + i] = make_float4(v.x, c, c, v.y);
                }
            }
        }
        __syncthreads();
        dst += (int64_t)w[l] * h[l];
    }
}

// The small end of the chain in one work group: every level from one of at
// most kTailTexels texels down to 1x1, level after level, each read back
// from the chain buffer that this work group wrote before the barrier.  The
// per-texel arithmetic is the blocks'; the levels cost one launch instead of
// one each (they are bound by launch latency, not by bytes).
constexpr int kTailThreads = 1024;
constexpr int kTailTexels = 64 * 64;

__global__ void __launch_bounds__(kTailThreads)
k_mip_tail(const float4* src, int ws, int hs, float4* dst) {
    while (ws > 1 || hs > 1) {
        const int wd = ws / 2 > 0 ? ws / 2 : 1, hd = hs / 2 > 0 ? hs / 2 : 1;
        for (int k = threadIdx.x; k < wd * hd; k += kTailThreads) {
            const int j = k / wd, i = k - j * wd;
            int x0, x1, y0, y1;
            float tx, ty;
            mip_axis(i, ws, wd, x0, x1, tx);
            mip_axis(j, hs, hd, y0, y1, ty);
            const float4 s00 = src[y0 * ws + x0], s01 = src[y0 * ws + x1];
            const float4 s10 = src[y1 * ws + x0], s11 = src[y1 * ws + x1];
            dst[k] = make_float4(bilerp(s00.x, s01.x, s10.x, s11.x, tx, ty),
                                 bilerp(s00.y, s01.y, s10.y, s11.y, tx, ty),
                                 bilerp(s00.z, s01.z, s10.z, s11.z, tx, ty),
                                 bilerp(s00.w, s01.w, s10.w, s11.w, tx, ty));
        }
        __syncthreads();  // this level is complete and visible to the whole group
        src = dst;
        dst += wd * hd;
        ws = wd;
        hs = hd;
    }
}

}  // namespace

int mip_chain(int W, int H, int* levels, size_t* floats) {
    int n = 0;
    for (int w = W, h = H; w > 0 || h > 0; w /= 2, h /= 2) ++n;
    size_t total = 0;
    for (int l = 1; l < n; ++l) {
        const size_t w = (size_t)(W >> l > 0 ? W >> l : 1), h = (size_t)(H >> l > 0 ? H >> l : 1);
        total += 4 * w * h;
    }
    if (levels) *levels = n;
    if (floats) *floats = total;
    return TWS_OK;
}

int grid_mips(GridState& g, float gb_fill, float* dst, size_t capacity_floats, hipStream_t s) {
    int levels = 0;
    size_t need = 0;
    mip_chain(g.W, g.H, &levels, &need);
    if (capacity_floats < need)
        return fail(TWS_ERR_INVALID, "mips: buffer holds %zu floats, the chain needs %zu",
                    capacity_floats, need);
    if (!std::isfinite(gb_fill)) return fail(TWS_ERR_INVALID, "mips: non-finite fill value");
    if (need > 0 && (!dst || reinterpret_cast<uintptr_t>(dst) % 16 != 0))
        return fail(TWS_ERR_INVALID, "mips: output must be a 16-byte aligned device buffer");
    const GridDesc gd = g.desc();
    float4* out = reinterpret_cast<float4*>(dst);
    const float4* prev = nullptr;
    int ws = g.W, hs = g.H;
    for (int left = levels - 1; left > 0;) {
        if (prev && ws * (int64_t)hs <= kTailTexels) {
            hipLaunchKernelGGL(k_mip_tail, dim3(1), dim3(kTailThreads), 0, s, prev, ws, hs, out);
            left = 0;
        } else {
            // Four levels where that leaves no more than the tail takes, else three:
            // as many launches up to 8192^2, and a block of an odd side computes
            // 35 x 35 texels of its first level instead of 39 x 39.  us a chain at
            // 4059 x 5027, with four levels and with three: 82.0 and
            // 77.6 (a launch per level: 76.0); 4096^2 58.5 -> 47.6 against that, 1024^2
            // 17.5 -> 10.9, 256^2 10.4 -> 9.1.
            int n = left < kMipLevels ? left : kMipLevels;
            if (n == kMipLevels && (int64_t)(ws >> n) * (hs >> n) > kTailTexels) n = kMipLevels - 1;
            // a small grid has too few blocks of four levels: two, the tail does the rest
            // (us a chain, four and two: 64^2 7.4, 6.8; 142 x 136 9.4, 8.5; 192^2 8.8, 8.3)
            if (!prev && n > 2 && (int64_t)ws * hs <= 192 * 192) n = 2;
            const int side = kMipSide >> (n - 1);
            const int wl = ws >> n > 0 ? ws >> n : 1, hl = hs >> n > 0 ? hs >> n : 1;
            const dim3 grid((wl + side - 1) / side, (hl + side - 1) / side);
            if (prev)
                hipLaunchKernelGGL((k_mip_block<false>), grid, dim3(kWave * kMipRows), 0, s, gd,
                                   g.parity, gb_fill, prev, ws, hs, out, n);
            else
                hipLaunchKernelGGL((k_mip_block<true>), grid, dim3(kWave * kMipRows), 0, s, gd,
                                   g.parity, gb_fill, prev, ws, hs, out, n);
            for (int l = 0; l < n; ++l) {
                prev = out;
                ws = ws / 2 > 0 ? ws / 2 : 1;
                hs = hs / 2 > 0 ? hs / 2 : 1;
                out += (size_t)ws * hs;
            }
            left -= n;
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(e, "mips: launch");
    }
    return TWS_OK;
}

}  // namespace tws
