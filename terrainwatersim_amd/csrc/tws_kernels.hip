// tws_kernels.hip -- gfx950 kernels of the virtual-pipe water step.
//
// Hot path: k_tile, the fused and temporally blocked step.  One work group
// owns an EXW x EXH tile of cells (the output tile plus a halo of 2 cells per
// step on each side) and advances it up to KH steps without touching HBM:
//   - each lane keeps CPL adjacent columns x RPW rows of depth d and flux f in
//     VGPRs for the whole launch; terrain b sits in LDS;
//   - x-neighbours come from the adjacent lane through DPP wave shifts,
//     y-neighbours from the lane's own registers, and only the first and last
//     row of each wave go through LDS;
//   - per step, two work-group barriers separate the flux phase
//     (flowUpdate.comp:29-62) from the depth phase (flowApply.comp:32-41).
// The halo region goes stale by 2 cells per step (flux needs h at radius 1,
// depth needs flux at radius 1), so after KH steps exactly the interior
// OX x OY cells are valid and stored.  HBM traffic per launch is one read of
// b, d, f and one write of d, f per output cell (plus the halo re-read),
// shared by KH steps.
//
// Every expression keeps the shaders' operation order and the library is
// compiled with -ffp-contract=off, so each cell's result is bit-identical to
// the FP32 restatement regardless of tile shape or steps per launch.

#include <algorithm>
#include <type_traits>

#include "tws_internal.hpp"
#include "tws.h"
#include "tws_fbm.hpp"
#include "tws_kernel_util.hpp"

namespace tws {

// ---------------------------------------------------------------------------
// What k_tile needs of a grid, in half a GridDesc: the planes lie one after the
// other (GridState::bind), so one pointer names them all.  A single-grid launch
// carries it by value, and the launch's start waits for those bytes: MI355X, ms
// per 1000 steps of the 256^2 rain grid (125 launches), 1.67 with 280 bytes of
// arguments, 1.645 with 236.
struct TileGrid {
    float* base;             // b | d0 | d1 | f0[4] | f1[4]
    unsigned int* status;
    int32_t pitch, W, H;
    int32_t tiles_x, tiles_y, tile_begin, tile_group;
    int32_t steps, parity0, boundary, rain_on, dry_ok;
    float F, K, C, ghost_alpha;
    float rain_cx, rain_cy, rain_I, rain_R2;

    __device__ __forceinline__ int64_t plane() const { return (int64_t)pitch * H; }
    __device__ __forceinline__ float* d(int set) const { return base + plane() * (1 + set); }
    __device__ __forceinline__ float* f(int set, int ch) const {
        return base + plane() * (3 + 4 * set + ch);
    }
};
__host__ __device__ inline TileGrid tile_grid(const GridDesc& g) {
    return TileGrid{const_cast<float*>(g.b), g.status, (int32_t)g.pitch, g.W, g.H, g.tiles_x,
                    g.tiles_y, g.tile_begin, g.tile_group, g.steps, g.parity0, g.boundary,
                    g.rain_on, g.dry_ok, g.F, g.K, g.C, g.ghost_d, g.rain_cx, g.rain_cy, g.rain_I,
                    g.rain_R2};
}

struct OneGrid {
    static constexpr bool kTable = false, kLooks = false;
    TileGrid g;
};
struct GridTable {
    static constexpr bool kTable = true, kLooks = false;
    const GridDesc* grids;
    const int* hdr;
    int launch_idx;
};
template <class Base>
struct Looking : Base {
    static constexpr bool kLooks = true;
    DryMaps dry;
};

// Tile (tx, ty) of a grid's tile list position lt: groups of tile_group tile
// columns, row by row within a group, so the tiles in flight at once form a
// compact block whose shared halos meet in L2 (tile_group 0: row-major).
__device__ __forceinline__ void tile_coords(const TileGrid& g, int lt, int& tx, int& ty) {
    if (g.tile_group > 0) {
        const int per_group = g.tile_group * g.tiles_y;
        const int grp = lt / per_group, in_grp = lt - grp * per_group;
        const int first = grp * g.tile_group;
        const int gw = min(g.tiles_x - first, g.tile_group);
        ty = in_grp / gw;
        tx = first + (in_grp - ty * gw);
    } else {
        ty = lt / g.tiles_x;
        tx = lt - ty * g.tiles_x;
    }
}

// One tile: load its EXW x EXH block of state set `parity`, advance it
// `levels` steps, store the valid interior into the other set.  Returns
// whether this lane stored a non-finite value.  MODE (kModePlain, kModeRain,
// kModeGeneral, kModeTruncated) compiles in only what the launch's grids use:
// the plain kernel has neither the rain source nor the reference-edge
// masking (no per-cell domain masks, so no scalar spills and 111 instead of
// 128 VGPRs at 128x64: +2.6% at k = 4, +7% at k = 6); the rain kernel has
// the rain but not the edge masking (6 instead of 23 scalar spills: +0.6% to
// +1.8% on closed-wall grids with rain).
// DRY: a tile is passed over while both buffer sets hold zeros there and
// nothing wet is within its halo, i.e. in the tiles around (DryMaps).  A kernel
// of its own: the code alone makes a launch of one tile per compute unit 4%
// longer (256^2), waiting for the marks one of a single round of work groups
// 5% (1500 x 1000).
template <int CPL, int RPW, int NW, int KH, int MODE, bool DRY>
__device__ __forceinline__ bool tile_step(const TileGrid& g, int tx, int ty, int levels,
                                          int parity, const uint8_t* dry_in,
                                          uint8_t* dry_out) {
    constexpr bool GEN = MODE != kModePlain;   // rain source compiled in
    constexpr bool EDGE = MODE >= kModeGeneral;  // reference-edge masking compiled in
    constexpr bool TAIL = MODE == kModeTruncated;  // cells no reference work group covers
    using G = TileGeom<CPL, RPW, NW, KH>;
    constexpr int EXW = G::EXW, EXH = G::EXH;
    __shared__ float s_b[EXH * EXW];
    __shared__ float s_xh[2][NW][CPL][kWave];  // [0]: first row of a wave, [1]: last row
    __shared__ float s_xf[2][NW][CPL][kWave];

    const int ox = tx * G::OX - G::HALOX;
    const int oy = ty * G::OY - G::HALOY;
    const int W = g.W, H = g.H;
    const int64_t pitch = g.pitch;
    const float F = g.F, K = g.K, C = g.C;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lx = lane * CPL;   // tile-local column of this lane's first cell
    const int ly = wave * RPW;   // tile-local row of this wave's first row
    const int x0 = ox + lx;
    float d[RPW][CPL], f0[RPW][CPL], f1[RPW][CPL], f2[RPW][CPL], f3[RPW][CPL];
    // ghost cells: closed walls, or the reference's out-of-image reads
    const bool closed = !EDGE || g.boundary == TWS_BOUNDARY_CLOSED;
    const float ghost_b = closed ? kWallHeight : 0.0f;
    const float ghost_d = closed ? 0.0f : g.ghost_alpha, ghost_fw = ghost_d;
    unsigned inside = 0;  // bit r*CPL+c: cell inside the domain
    // The same for the cells the reference's truncating dispatch shapes leave as
    // they are, and those its brush covers (GridDesc::upd_w, brush_w).
    unsigned frozen = 0, brushed = 0;
    const bool tail = TAIL && (ox + EXW > (W & ~15) || oy + EXH > (H & ~15));
    bool bad = false;

    // The marks of this tile and the tiles around it: lane i < 9 reads those of
    // neighbour (i % 3 - 1, i / 3 - 1).
    static_assert(NW == 8 || NW == 16, "a tile's marks are one or two 8-byte words");
    constexpr int kWords = NW / 8;
    constexpr uint64_t kOnes = 0x0101010101010101ull;
    const int64_t marks_at = g.tile_begin + ty * g.tiles_x + tx;
    bool before = false;  // this wavefront's output was dry in the launch before
    if constexpr (DRY)
        if (dry_in) {
            const int nx = tx + lane % 3 - 1, ny = ty + lane / 3 - 1;
            bool around = true;
            if (lane < 9 && nx >= 0 && nx < g.tiles_x && ny >= 0 && ny < g.tiles_y)
#pragma unroll
                for (int i = 0; i < kWords; ++i) {
                    const uint64_t m = reinterpret_cast<const uint64_t*>(
                        dry_in)[(g.tile_begin + ny * g.tiles_x + nx) * (int64_t)kWords + i];
                    around = around && (lane == 4 ? (m & 2 * kOnes) == 2 * kOnes
                                                  : ((m | m >> 1) & kOnes) == kOnes);
                    if (lane == 4 && i == wave / 8) before = (m >> (wave % 8 * 8) & 3) != 0;
                }
            before = __ballot(before) != 0;
            // the rain on any wavefront's rows keeps the whole tile
            if (__ballot(!around) == 0 &&
                !(GEN && g.rain_on != 0 &&
                  __builtin_amdgcn_readfirstlane(brush_reaches(g.rain_cx, g.rain_cy, g.rain_R2, ox,
                                                               ox + EXW - 1, oy, oy + EXH - 1)
                                                     ? 1 : 0) != 0)) {
                if (lane == 0) dry_out[marks_at * NW + wave] = 2;
                return false;  // every wavefront of the group alike
            }
        }

    // ---- load -------------------------------------------------------------
    // All loads of the wavefront are issued before the first is waited for, the
    // terrain first: no branch surrounds them, from addresses clamped into the
    // grid, and what lies outside it is replaced afterwards.  (A branch per row
    // had every row wait for the one before, RPW round trips to memory.  MI355X,
    // us before -> after: 1500 x 1000 sheet, 100 steps, 624 -> 588; 2048^2 with a
    // lake, 100 steps, 1100 -> 1020; 256^2 rain, 1000 steps, 1596 -> 1562; 4096^2
    // zero edge all wet, 96 steps, 4490 -> 4300.)
    const bool edge_tile = ox < 0 || oy < 0 || ox + EXW > W || oy + EXH > H;
    float vb[RPW][CPL];
    {
        // A row's address is wave-uniform.  Lanes of 16 cells, whose vector
        // registers the loads fill, keep it in scalar ones; the others, whose
        // residency many scalar registers cost, an offset from their first row's.
        constexpr bool kRowScalar = CPL * RPW >= 16;
        const int top = kRowScalar ? 0 : min(max(oy + ly, 0), H - 1);
        const uint32_t xb = (uint32_t)min(max(x0, 0), g.pitch - CPL) * 4u;
        auto load = [&](const float* plane, float (&v)[RPW][CPL]) {
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                const int row = min(max(oy + ly + r, 0), H - 1) - top;
                if constexpr (kRowScalar) vload<CPL>(at(plane, row * pitch, xb), v[r]);
                else vload<CPL>(at(plane, top * pitch, xb + (uint32_t)row * (uint32_t)g.pitch * 4u), v[r]);
            }
        };
        load(g.base, vb);
        load(g.d(parity), d);
        load(g.f(parity, 0), f0);
        load(g.f(parity, 1), f1);
        load(g.f(parity, 2), f2);
        load(g.f(parity, 3), f3);
    }
    // The brush amounts do not change from level to level: computed once, in
    // registers across the loop (recomputing them per level measured 13%
    // slower at 256^2, where waves under the disc are on the critical path),
    // and only by waves under the disc.  Left to itself the compiler hoisted
    // the divisions out of the loop into every wave.  While the loads are on
    // their way, but for lanes of 16 cells, which have no registers to spare until
    // the terrain is in LDS (3001 x 2777 zero edge, 60 steps: 1538 us against 1349).
    // A wave whose rows lie wholly outside the disc skips the brush (wave-uniform).
    float wet[RPW][CPL];
    bool rain = false;
    auto brush = [&]() {
        rain = GEN && g.rain_on != 0 &&
               __builtin_amdgcn_readfirstlane(brush_reaches(g.rain_cx, g.rain_cy, g.rain_R2, ox,
                                                            ox + EXW - 1, oy + ly,
                                                            oy + ly + RPW - 1)
                                                  ? 1 : 0) != 0;
        if (rain) {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    wet[r][c] = brush_amount(g.rain_cx, g.rain_cy, g.rain_I, g.rain_R2, x0 + c,
                                             oy + ly + r);
        } else {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int c = 0; c < CPL; ++c) wet[r][c] = 0.0f;
        }
    };
    constexpr bool kBrushEarly = CPL * RPW < 16;
    if constexpr (kBrushEarly) brush();
    // The tile's cells outside the grid become ghosts.
    auto in_grid = [&](int r, int c) {
        return (unsigned)(oy + ly + r) < (unsigned)H && (unsigned)(x0 + c) < (unsigned)W;
    };
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const bool in = in_grid(r, c);
            inside |= (in ? 1u : 0u) << (r * CPL + c);
            if constexpr (TAIL) {
                const int x = x0 + c, y = oy + ly + r;
                frozen |= (in && (x >= (W & ~15) || y >= (H & ~15)) ? 1u : 0u) << (r * CPL + c);
                brushed |= (in && x < (W & ~31) && y < (H & ~31) ? 1u : 0u) << (r * CPL + c);
            }
        }
    if (edge_tile) {
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const bool in = in_grid(r, c);
                vb[r][c] = in ? vb[r][c] : ghost_b;
                d[r][c] = in ? d[r][c] : ghost_d;
                f0[r][c] = in ? f0[r][c] : 0.0f;
                f1[r][c] = in ? f1[r][c] : 0.0f;
                f2[r][c] = in ? f2[r][c] : 0.0f;
                f3[r][c] = in ? f3[r][c] : ghost_fw;
            }
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c) s_b[(ly + r) * EXW + lx + c] = vb[r][c];
    const bool need_mask = EDGE && g.boundary != TWS_BOUNDARY_CLOSED && edge_tile;
    // Closed walls carry no flux either way.  The wall ghost makes every
    // wall-ward flux the kernel computes max(0, f*F + (h - 1e30)*K) = +0 as
    // long as the cell's own stored wall-ward f is 0; an uploaded state may
    // hold another value there (and with K = 0 it would pass the wall), so
    // edge cells drop it as they load.
    if ((!EDGE || g.boundary == TWS_BOUNDARY_CLOSED) && edge_tile) {
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const int y = oy + ly + r;
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const int x = x0 + c;
                if (x == W - 1) f0[r][c] = 0.0f;
                if (x == 0) f1[r][c] = 0.0f;
                if (y == H - 1) f2[r][c] = 0.0f;
                if (y == 0) f3[r][c] = 0.0f;
            }
        }
    }
    if constexpr (!kBrushEarly) brush();
    __syncthreads();  // s_b complete

    for (int lev = 0; lev < levels; ++lev) {
        if (rain) {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if ((TAIL ? brushed : inside) & (1u << (r * CPL + c)))
                        d[r][c] = d[r][c] + wet[r][c];
        }

        // ---- flux phase: flowUpdate.comp:34-62 ------------------------------
        float h[RPW][CPL];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) h[r][c] = d[r][c] + s_b[(ly + r) * EXW + lx + c];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            s_xh[0][wave][c][lane] = h[0][c];
            s_xh[1][wave][c][lane] = h[RPW - 1][c];
        }
        __syncthreads();
        float h_up[CPL], h_dn[CPL];  // rows y-1 of the first row and y+1 of the last row
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            h_up[c] = wave > 0 ? s_xh[1][wave - 1][c][lane] : h[0][c];
            h_dn[c] = wave < NW - 1 ? s_xh[0][wave + 1][c][lane] : h[RPW - 1][c];
        }
        // Rows that can still reach the output: the flux of level lev is
        // needed on rows [2 lev + 1, EXH - 2 lev - 1), the depth on
        // [2 lev + 2, EXH - 2 lev - 2).  Rows outside only feed rows outside,
        // so a wave may skip them (wave-uniform branches).  Measured: +12-14%
        // for 64x64 tiles at 256^2-512^2, +2-5% for the general kernel at
        // 2048^2-4096^2, but -2% for the plain kernels whose lanes hold 16
        // cells (the branches cost more than the rows they save there).
        constexpr bool kSkipRows = GEN || CPL * RPW < 16;
        const int flo = 2 * lev + 1 - ly, fhi = EXH - 2 * lev - 1 - ly;
        const bool live = lane_in(live_lanes<CPL>(lev));
        // Each head difference, times K, serves the two cells it separates
        // (negated for the second: fl(a - b) = -fl(b - a) exactly).  The lane past
        // the tile's edge reads as 0, whatever that makes of the edge column, and
        // only live lanes ask for the division.  5.5 of 47 vector instructions a
        // cell and level fewer (64x64); MI355X, us before -> after: 256^2 rain, 1000
        // steps, 1637 -> 1599; 2048^2 with a lake, 100 steps, 1141 -> 1091; 3001 x
        // 2777 zero edge, 60 steps, 1423 -> 1396; 1500 x 1000, 100 steps, 629 -> 624.
        // (k_stream's registers are full: the masks cost its 4096^2 sheet 2%.)
        float py_up[CPL];  // of rows r-1 and r
#pragma unroll
        for (int c = 0; c < CPL; ++c) py_up[c] = (h_up[c] - h[0][c]) * K;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            float py[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c)
                py[c] = (h[r][c] - (r < RPW - 1 ? h[r + 1][c] : h_dn[c])) * K;
            if (!kSkipRows || (r >= flo && r < fhi)) {
                const float h_right = from_right_lane(h[r][0]);
                float px[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    px[c] = (h[r][c] - (c < CPL - 1 ? h[r][c + 1] : h_right)) * K;
                const float px_left = from_left_lane(px[CPL - 1]);
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    const float k0 = f0[r][c], k1 = f1[r][c], k2 = f2[r][c], k3 = f3[r][c];
                    flux_update_p(F, C, d[r][c], live, px[c], -(c > 0 ? px[c - 1] : px_left), py[c],
                                  -py_up[c], f0[r][c], f1[r][c], f2[r][c], f3[r][c]);
                    if (TAIL && tail && (frozen & (1u << (r * CPL + c)))) {
                        f0[r][c] = k0; f1[r][c] = k1; f2[r][c] = k2; f3[r][c] = k3;
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < CPL; ++c) py_up[c] = py[c];
        }
        if (need_mask) {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if (!(inside & (1u << (r * CPL + c)))) {
                        f0[r][c] = 0.0f; f1[r][c] = 0.0f; f2[r][c] = 0.0f;
                        f3[r][c] = ghost_fw;
                    }
        }

        // ---- depth phase: flowApply.comp:32-41 -------------------------------
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            s_xf[0][wave][c][lane] = f3[0][c];        // -y flux of the first row
            s_xf[1][wave][c][lane] = f2[RPW - 1][c];  // +y flux of the last row
        }
        __syncthreads();
        float f_up[CPL], f_dn[CPL];  // +y flux of row y-1, -y flux of row y+1
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            f_up[c] = wave > 0 ? s_xf[1][wave - 1][c][lane] : 0.0f;
            f_dn[c] = wave < NW - 1 ? s_xf[0][wave + 1][c][lane] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            if (kSkipRows && (r < flo + 1 || r >= fhi - 1)) continue;
            const float in_left = from_left_lane(f0[r][CPL - 1]);   // X0.x
            const float in_right = from_right_lane(f1[r][0]);      // X1.y
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const float X1y = c < CPL - 1 ? f1[r][c + 1] : in_right;
                const float X0x = c > 0 ? f0[r][c - 1] : in_left;
                const float Y1w = r < RPW - 1 ? f3[r + 1][c] : f_dn[c];
                const float Y0z = r > 0 ? f2[r - 1][c] : f_up[c];
                const float in = ((X1y + X0x) + Y1w) + Y0z;
                const float out = ((f0[r][c] + f1[r][c]) + f2[r][c]) + f3[r][c];
                const float nd = fmaxf(0.0f, d[r][c] + (in - out) * C);
                if (!(TAIL && tail && (frozen & (1u << (r * CPL + c))))) d[r][c] = nd;
            }
        }
        if (need_mask) {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if (!(inside & (1u << (r * CPL + c)))) d[r][c] = ghost_d;
        }
    }

    // ---- store the valid interior ------------------------------------------
    {
        gfloat* __restrict__ pd = gptr(g.d(parity ^ 1));
        gfloat* __restrict__ p0 = gptr(g.f(parity ^ 1, 0));
        gfloat* __restrict__ p1 = gptr(g.f(parity ^ 1, 1));
        gfloat* __restrict__ p2 = gptr(g.f(parity ^ 1, 2));
        gfloat* __restrict__ p3 = gptr(g.f(parity ^ 1, 3));
        const bool col_ok = lx >= G::HALOX && lx < EXW - G::HALOX && x0 < W;
        const bool full = x0 + CPL <= W;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const int yl = ly + r;
            const int y = oy + yl;
            if (!(col_ok && yl >= G::HALOY && yl < EXH - G::HALOY && y < H)) continue;
            const int64_t off = (int64_t)y * pitch + x0;
#pragma unroll
            for (int c = 0; c < CPL; ++c)
                bad |= (full || x0 + c < W) &
                       nonfinite5(d[r][c], f0[r][c], f1[r][c], f2[r][c], f3[r][c]);
            if (full) {
                vstore<CPL>(pd + off, d[r]);
                vstore<CPL>(p0 + off, f0[r]);
                vstore<CPL>(p1 + off, f1[r]);
                vstore<CPL>(p2 + off, f2[r]);
                vstore<CPL>(p3 + off, f3[r]);
            } else {
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if (x0 + c < W) {
                        pd[off + c] = d[r][c];
                        p0[off + c] = f0[r][c];
                        p1[off + c] = f1[r][c];
                        p2[off + c] = f2[r][c];
                        p3[off + c] = f3[r][c];
                    }
            }
        }
        if constexpr (DRY) {
            unsigned held = 0;  // bits of the lane's output
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                const int yl = ly + r;
                if (!(col_ok && yl >= G::HALOY && yl < EXH - G::HALOY && oy + yl < H)) continue;
#pragma unroll
                for (int c = 0; c < CPL; ++c)
                    if (full || x0 + c < W)
                        held |= __float_as_uint(d[r][c]) | __float_as_uint(f0[r][c]) |
                                __float_as_uint(f1[r][c]) | __float_as_uint(f2[r][c]) |
                                __float_as_uint(f3[r][c]);
            }
            bool dry = g.dry_ok != 0 && __ballot(held != 0) == 0;
            if (dry) {  // on ground where dry cells stay dry
                bool ok = true;
                for (int r = 0; r < RPW; ++r) {
                    const int yl = ly + r;
                    if (!(col_ok && yl >= G::HALOY && yl < EXH - G::HALOY && oy + yl < H)) continue;
                    for (int c = 0; c < CPL; ++c)
                        ok = ok && (x0 + c >= W || regular_height(s_b[yl * EXW + lx + c]));
                }
                dry = __ballot(!ok) == 0;
            }
            if (lane == 0) dry_out[marks_at * NW + wave] = dry ? (before ? 2 : 1) : 0;
        }
    }
    return bad;
}

// ---------------------------------------------------------------------------
// Fused, temporally blocked step.  Grid: one block per tile of the flattened
// tile list; blocks past the tile count exit at once.  The arguments are of the
// launch's kind, since a launch of one round of tiles notices their size (a 256^2
// rain grid at k = 8, us per launch: 13.35 with 108 bytes, 13.50 with 124):
//   OneGrid    the grid by value;
//   GridTable  hdr = {number of grids, number of tiles, offset} and
//              grids[offset..] (ordered by tile_begin) in device memory, so a
//              captured launch stays valid while grids come and go;
//   Looking    either, looking for dry tiles.  MODE is the highest kernel_mode of the launch's grids
// (chosen on the host from the descriptors).
// At least 4 waves per SIMD (at most 128 VGPRs): 2 work groups of 512 per CU.
template <int CPL, int RPW, int NW, int KH, int MODE, class Args>
__global__ void __launch_bounds__(NW * kWave, 4)
k_tile(Args args) {
    constexpr bool DRY = Args::kLooks;
    // XCD-aware order: the hardware deals blocks to the 8 XCDs round robin;
    // give each XCD a contiguous run of tiles so neighbouring tiles (whose
    // halos overlap) share one L2.
    int total_tiles;
    if constexpr (Args::kTable) total_tiles = args.hdr[1];
    else total_tiles = args.g.tiles_x * args.g.tiles_y;
    const int bid = blockIdx.x;
    if (Args::kTable && bid >= total_tiles) return;
    const int xcd = bid & 7, idx = bid >> 3;
    const int q = total_tiles >> 3, rmd = total_tiles & 7;
    int tile = xcd * q + (xcd < rmd ? xcd : rmd) + idx;
    if constexpr (DRY) {
        // Runs of 32 tiles only, dealt round the XCDs: water gathers in some
        // part of a grid, and an XCD with a whole eighth of the tiles would
        // step it alone (2048^2 with a lake over 27% of the tiles: 48 us a
        // launch with eighths).
        constexpr int kRun = 32;
        const int dealt = total_tiles / (8 * kRun) * (8 * kRun);
        tile = bid < dealt ? (idx / kRun * 8 + xcd) * kRun + idx % kRun : bid;
    }

    TileGrid g;
    int launch_idx = 0;
    if constexpr (Args::kTable) {
        const GridDesc* grids = args.grids + args.hdr[2];  // this launch's segment of the table
        launch_idx = args.launch_idx;
        int lo = 0, hi = args.hdr[0] - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (grids[mid].tile_begin <= tile) lo = mid; else hi = mid - 1;
        }
        g = tile_grid(grids[lo]);
    } else {
        g = args.g;
    }
    const int levels = min(KH, g.steps - launch_idx * KH);
    if (Args::kTable && levels <= 0) return;
    const int parity = (g.parity0 + launch_idx) & 1;
    // Every other launch walks the grid's tiles backwards, so it starts on the
    // tiles the launch before wrote last, whose state may still sit in the
    // memory-side cache.  Tiles of one launch are independent: the order does
    // not change results.
    int lt = tile - g.tile_begin;
    if (parity) lt = g.tiles_x * g.tiles_y - 1 - lt;
    int tx, ty;
    tile_coords(g, lt, tx, ty);
    const uint8_t* dry_in = nullptr;
    uint8_t* dry_out = nullptr;
    if constexpr (DRY) {
        dry_in = args.dry.in;
        dry_out = args.dry.out;
    }
    const bool bad = tile_step<CPL, RPW, NW, KH, MODE, DRY>(g, tx, ty, levels, parity, dry_in,
                                                            dry_out);
    if (__ballot(bad) != 0 && (threadIdx.x & (kWave - 1)) == 0) atomicOr(g.status, 1u);
}

// ---------------------------------------------------------------------------
// Two-pass step with the reference's structure: a flux kernel and an apply
// kernel per step, neighbours read from memory.  Reads set `parity`, writes
// flux to set parity^1 (flux pass) and depth to set parity^1 (apply pass).
__global__ void __launch_bounds__(256) k_flux_twopass(GridDesc g, int parity) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t p = g.pitch, i = (int64_t)y * p + x;
    if (x >= g.upd_w || y >= g.upd_h) {  // no reference work group covers it
        for (int c = 0; c < 4; ++c) g.f[parity ^ 1][c][i] = g.f[parity][c][i];
        return;
    }
    const float* b = g.b;
    const float* d = g.d[parity];
    const bool in_x1 = x + 1 < g.W, in_x0 = x > 0, in_y1 = y + 1 < g.H, in_y0 = y > 0;
    const float gh = g.ghost_d + g.ghost_b;  // never used in closed mode
    const float own = d[i] + b[i];
    const float hx1 = in_x1 ? d[i + 1] + b[i + 1] : gh;
    const float hx0 = in_x0 ? d[i - 1] + b[i - 1] : gh;
    const float hy1 = in_y1 ? d[i + p] + b[i + p] : gh;
    const float hy0 = in_y0 ? d[i - p] + b[i - p] : gh;
    float o0 = g.f[parity][0][i], o1 = g.f[parity][1][i], o2 = g.f[parity][2][i],
          o3 = g.f[parity][3][i];
    if (g.boundary == TWS_BOUNDARY_CLOSED) {
        // the flux toward a wall is clamped to zero before the scaling sum
        float t0 = fmaxf(0.0f, o0 * g.F + (own - hx1) * g.K);
        float t1 = fmaxf(0.0f, o1 * g.F + (own - hx0) * g.K);
        float t2 = fmaxf(0.0f, o2 * g.F + (own - hy1) * g.K);
        float t3 = fmaxf(0.0f, o3 * g.F + (own - hy0) * g.K);
        if (!in_x1) t0 = 0.0f;
        if (!in_x0) t1 = 0.0f;
        if (!in_y1) t2 = 0.0f;
        if (!in_y0) t3 = 0.0f;
        const float total = ((t0 + t1) + (t2 + t3)) * g.C;
        if (total > d[i]) {
            const float s = d[i] / total;
            t0 = t0 * s; t1 = t1 * s; t2 = t2 * s; t3 = t3 * s;
        }
        o0 = t0; o1 = t1; o2 = t2; o3 = t3;
    } else {
        flux_update(g.F, g.K, g.C, d[i], own - hx1, own - hx0, own - hy1, own - hy0, o0, o1, o2,
                    o3);
    }
    g.f[parity ^ 1][0][i] = o0;
    g.f[parity ^ 1][1][i] = o1;
    g.f[parity ^ 1][2][i] = o2;
    g.f[parity ^ 1][3][i] = o3;
}

__global__ void __launch_bounds__(256) k_apply_twopass(GridDesc g, int parity) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t p = g.pitch, i = (int64_t)y * p + x;
    if (x >= g.upd_w || y >= g.upd_h) {  // no reference work group covers it
        g.d[parity ^ 1][i] = g.d[parity][i];
        return;
    }
    float* const* fo = g.f[parity ^ 1];
    const float gz = g.boundary == TWS_BOUNDARY_CLOSED ? 0.0f : g.ghost_fw;
    const float X1y = x + 1 < g.W ? fo[1][i + 1] : 0.0f;
    const float X0x = x > 0 ? fo[0][i - 1] : 0.0f;
    const float Y1w = y + 1 < g.H ? fo[3][i + p] : gz;
    const float Y0z = y > 0 ? fo[2][i - p] : 0.0f;
    const float in = ((X1y + X0x) + Y1w) + Y0z;
    const float out = ((fo[0][i] + fo[1][i]) + fo[2][i]) + fo[3][i];
    g.d[parity ^ 1][i] = fmaxf(0.0f, g.d[parity][i] + (in - out) * g.C);
}

// One brush application to the depth plane of set `parity`, in place.
__global__ void __launch_bounds__(256) k_brush(GridDesc g, int parity, float cx, float cy,
                                                float I, float R2) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.brush_w || y >= g.brush_h) return;
    const int64_t i = (int64_t)y * g.pitch + x;
    float* d = g.d[parity];
    d[i] = d[i] + brush_amount(cx, cy, I, R2, x, y);
}

// Directed flow from the current flux, flowApply.comp:45-46; dense output
// v2[(x + y*W)*2 + {0,1}].
__global__ void __launch_bounds__(256) k_velocity(GridDesc g, int parity, float* v2) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t p = g.pitch, i = (int64_t)y * p + x;
    float* const* f = g.f[parity];
    const float gz = g.boundary == TWS_BOUNDARY_CLOSED ? 0.0f : g.ghost_fw;
    const float X1y = x + 1 < g.W ? f[1][i + 1] : 0.0f;
    const float X0x = x > 0 ? f[0][i - 1] : 0.0f;
    const float Y1w = y + 1 < g.H ? f[3][i + p] : gz;
    const float Y0z = y > 0 ? f[2][i - p] : 0.0f;
    const int64_t o = (int64_t)y * g.W + x;
    // a cell no reference work group covers never receives a FlowMap value
    const bool upd = x < g.upd_w && y < g.upd_h;
    v2[o * 2 + 0] = upd ? (X1y - f[0][i]) - (X0x - f[1][i]) : 0.0f;
    v2[o * 2 + 1] = upd ? (Y1w - f[2][i]) - (Y0z - f[3][i]) : 0.0f;
}

// Planar flux of set `parity` <-> dense interleaved staging[(x + y*W)*4 + c].
__global__ void __launch_bounds__(256) k_interleave(GridDesc g, int parity, float* st) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t i = (int64_t)y * g.pitch + x, o = (int64_t)y * g.W + x;
    *reinterpret_cast<float4*>(st + o * 4) =
        make_float4(g.f[parity][0][i], g.f[parity][1][i], g.f[parity][2][i], g.f[parity][3][i]);
}
__global__ void __launch_bounds__(256) k_deinterleave(GridDesc g, int parity, const float* st) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t i = (int64_t)y * g.pitch + x, o = (int64_t)y * g.W + x;
    const float4 v = *reinterpret_cast<const float4*>(st + o * 4);
    g.f[parity][0][i] = v.x; g.f[parity][1][i] = v.y;
    g.f[parity][2][i] = v.z; g.f[parity][3][i] = v.w;
}

// Reference interleaved layout (Terrain.cpp:205-237) -> planes.
__global__ void __launch_bounds__(256) k_ref_unpack(GridDesc g, int parity, const float* terrain,
                                                     const float* flow, float* b_out) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t i = (int64_t)y * g.pitch + x, o = (int64_t)y * g.W + x;
    if (terrain) {
        const float4 t = *reinterpret_cast<const float4*>(terrain + o * 4);
        b_out[i] = t.x;
        g.d[parity][i] = t.w;
    }
    if (flow) {
        const float4 v = *reinterpret_cast<const float4*>(flow + o * 4);
        g.f[parity][0][i] = v.x; g.f[parity][1][i] = v.y;
        g.f[parity][2][i] = v.z; g.f[parity][3][i] = v.w;
    }
}

// Planes -> reference layout; FlowMap as rg16f bits (flowApply.comp:52).
__global__ void __launch_bounds__(256) k_ref_pack(GridDesc g, int parity, float gb_fill,
                                                   float* terrain, float* flow, uint16_t* flowmap) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t p = g.pitch, i = (int64_t)y * p + x, o = (int64_t)y * g.W + x;
    float* const* f = g.f[parity];
    if (terrain)
        *reinterpret_cast<float4*>(terrain + o * 4) = make_float4(g.b[i], gb_fill, gb_fill, g.d[parity][i]);
    if (flow)
        *reinterpret_cast<float4*>(flow + o * 4) = make_float4(f[0][i], f[1][i], f[2][i], f[3][i]);
    if (flowmap) {
        const float gz = g.boundary == TWS_BOUNDARY_CLOSED ? 0.0f : g.ghost_fw;
        const float X1y = x + 1 < g.W ? f[1][i + 1] : 0.0f;
        const float X0x = x > 0 ? f[0][i - 1] : 0.0f;
        const float Y1w = y + 1 < g.H ? f[3][i + p] : gz;
        const float Y0z = y > 0 ? f[2][i - p] : 0.0f;
        const bool upd = x < g.upd_w && y < g.upd_h;  // see k_velocity
        flowmap[o * 2 + 0] = upd ? half_rtz((X1y - f[0][i]) - (X0x - f[1][i])) : (uint16_t)0;
        flowmap[o * 2 + 1] = upd ? half_rtz((Y1w - f[2][i]) - (Y0z - f[3][i])) : (uint16_t)0;
    }
}

// FP64 partial sums of depth: block p takes rows p, p+nparts, ...; threads
// stride the columns; a fixed tree combines them.  Deterministic.
__global__ void __launch_bounds__(256) k_volume(GridDesc g, int parity, double* partials,
                                                 int nparts) {
    __shared__ double s[256];
    double acc = 0.0;
    const float* d = g.d[parity];
    for (int y = blockIdx.x; y < g.H; y += nparts)
        for (int x = threadIdx.x; x < g.W; x += 256) acc += (double)d[(int64_t)y * g.pitch + x];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = s[0];
}

__global__ void __launch_bounds__(256) k_zero_fill(float* p, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0.0f;
}

// Finiteness of the state of set `parity` (b, d, f) after an upload: sets
// bit 0 of *status if any value inside the domain is NaN or Inf.  The step
// kernel itself only checks what it stores (its max(0, .) clamps would turn
// a NaN input into 0).
__global__ void __launch_bounds__(256) k_check_finite(GridDesc g, int parity) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    bool bad = false;
    if (x < g.W && y < g.H) {
        const int64_t i = (int64_t)y * g.pitch + x;
        bad = nonfinite5(g.b[i], g.d[parity][i], g.f[parity][0][i], g.f[parity][1][i],
                         g.f[parity][2][i]) |
              !__builtin_isfinite(g.f[parity][3][i]);
    }
    if (__ballot(bad) != 0 && (threadIdx.x & 63) == 0) atomicOr(g.status, 1u);
}

// Seeded fBm terrain straight into the b plane (same bits as the host
// generator: tws_fbm.hpp).
__global__ void __launch_bounds__(256) k_fbm(float* b, int64_t pitch, int W, int H,
                                              uint64_t seed, int octaves, int base,
                                              double persistence, double scale) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= W || y >= H) return;
    b[(int64_t)y * pitch + x] = fbm_cell(x, y, W, H, seed, octaves, base, persistence, scale);
}

// Water of set `parity`: rect_depth inside [x0, x1) x [y0, y1), `depth`
// elsewhere; flux zero.
__global__ void __launch_bounds__(256) k_init_water(GridDesc g, int parity, float depth, int x0,
                                                     int y0, int x1, int y1, float rect_depth) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= g.W || y >= g.H) return;
    const int64_t i = (int64_t)y * g.pitch + x;
    const bool in = x >= x0 && x < x1 && y >= y0 && y < y1;
    g.d[parity][i] = in ? rect_depth : depth;
    for (int c = 0; c < 4; ++c) g.f[parity][c][i] = 0.0f;
}

// Device copy of n float4 (STREAM copy): the measured HBM ceiling, and the
// known-size reference that scales the FETCH_SIZE / WRITE_SIZE counters.
// Each lane keeps U loads in flight (issued back to back, then U stores);
// NT marks them non-temporal.  Chunks of U * blockDim float4 are dealt out
// grid-stride; the tail chunk is bounds-checked per element.
template <int U, bool NT>
__global__ void __launch_bounds__(256) k_stream_copy(const vf4* __restrict__ src,
                                                      vf4* __restrict__ dst, int64_t n) {
    const int64_t chunk = (int64_t)U * blockDim.x;
    for (int64_t base = (int64_t)blockIdx.x * chunk; base < n; base += (int64_t)gridDim.x * chunk) {
        vf4 v[U];
        if (base + chunk <= n) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = base + (int64_t)u * blockDim.x + threadIdx.x;
                v[u] = NT ? __builtin_nontemporal_load(src + i) : src[i];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = base + (int64_t)u * blockDim.x + threadIdx.x;
                if (NT) __builtin_nontemporal_store(v[u], dst + i); else dst[i] = v[u];
            }
        } else {
            for (int u = 0; u < U; ++u) {
                const int64_t i = base + (int64_t)u * blockDim.x + threadIdx.x;
                if (i < n) dst[i] = src[i];
            }
        }
    }
}

// Lane-layout check of the DPP wave shifts used by k_tile.
__global__ void __launch_bounds__(64) k_lane_shift_probe(int* out) {
    const int lane = threadIdx.x;
    // lane i holds i + 1, so a lane without a source (which reads 0) shows as 0
    out[lane] = __float_as_int(from_left_lane(__int_as_float(lane + 1)));
    out[64 + lane] = __float_as_int(from_right_lane(__int_as_float(lane + 1)));
}

// ---------------------------------------------------------------------------
// Host-side launch helpers.

static dim3 cell_grid(const GridDesc& g) { return dim3((g.W + 15) / 16, (g.H + 15) / 16); }

// Launches that look for dry tiles are built for the pairs the tile table
// gives grids of many tiles.
static constexpr bool dry_built(int cpl, int nw, int k) {
    return nw == 8 && (k == 4 || k == 5) && (cpl == 1 || cpl == 2);
}
bool tile_looks(int kernel, int k) {
    return (kernel == TWS_KERNEL_TILE_64x64 && dry_built(1, 8, k)) ||
           (kernel == TWS_KERNEL_TILE_128x64 && dry_built(2, 8, k));
}

template <int CPL, int RPW, int NW, int MODE, class Args>
static hipError_t launch_tile_kg(int k, const Args& args, int blocks, const DryMaps& dry,
                                 hipStream_t s) {
    const dim3 grid(blocks), block(NW * kWave);
    auto launch = [&](auto steps) {
        constexpr int KH = decltype(steps)::value;
        if constexpr (dry_built(CPL, NW, KH)) {
            if (dry.out) {
                Looking<Args> look;
                static_cast<Args&>(look) = args;
                look.dry = dry;
                hipLaunchKernelGGL((k_tile<CPL, RPW, NW, KH, MODE, Looking<Args>>), grid, block, 0,
                                   s, look);
                return hipGetLastError();
            }
        }
        if (dry.out) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_tile<CPL, RPW, NW, KH, MODE, Args>), grid, block, 0, s, args);
        return hipGetLastError();
    };
    switch (k) {
        case 1: return launch(std::integral_constant<int, 1>{});
        case 2: return launch(std::integral_constant<int, 2>{});
        case 3: return launch(std::integral_constant<int, 3>{});
        case 4: return launch(std::integral_constant<int, 4>{});
        case 5: return launch(std::integral_constant<int, 5>{});
        case 6: return launch(std::integral_constant<int, 6>{});
        case 8: return launch(std::integral_constant<int, 8>{});
        default: return hipErrorInvalidValue;
    }
}

template <int CPL, int RPW, int NW, class Args>
static hipError_t launch_tile_k(int k, int mode, const Args& args, int blocks, const DryMaps& dry,
                                hipStream_t s) {
    switch (mode) {
        case kModePlain: return launch_tile_kg<CPL, RPW, NW, kModePlain>(k, args, blocks, dry, s);
        case kModeRain: return launch_tile_kg<CPL, RPW, NW, kModeRain>(k, args, blocks, dry, s);
        case kModeGeneral: return launch_tile_kg<CPL, RPW, NW, kModeGeneral>(k, args, blocks, dry, s);
        default: break;
    }
    if constexpr (Args::kTable) return hipErrorInvalidValue;  // a batch takes no such grid
    else return launch_tile_kg<CPL, RPW, NW, kModeTruncated>(k, args, blocks, dry, s);
}

template <int CPL, int RPW, int NW>
static void shape_of(int k, TileShape* out) {
    int ox = 0, oy = 0;
    switch (k) {
        case 1: ox = TileGeom<CPL, RPW, NW, 1>::OX; oy = TileGeom<CPL, RPW, NW, 1>::OY; break;
        case 2: ox = TileGeom<CPL, RPW, NW, 2>::OX; oy = TileGeom<CPL, RPW, NW, 2>::OY; break;
        case 4: ox = TileGeom<CPL, RPW, NW, 4>::OX; oy = TileGeom<CPL, RPW, NW, 4>::OY; break;
        case 3: ox = TileGeom<CPL, RPW, NW, 3>::OX; oy = TileGeom<CPL, RPW, NW, 3>::OY; break;
        case 5: ox = TileGeom<CPL, RPW, NW, 5>::OX; oy = TileGeom<CPL, RPW, NW, 5>::OY; break;
        case 6: ox = TileGeom<CPL, RPW, NW, 6>::OX; oy = TileGeom<CPL, RPW, NW, 6>::OY; break;
        case 8: ox = TileGeom<CPL, RPW, NW, 8>::OX; oy = TileGeom<CPL, RPW, NW, 8>::OY; break;
    }
    out->ox = ox; out->oy = oy; out->threads = NW * kWave;
}

bool tile_shape(int kernel, int k, TileShape* out) {
    if (k < 1 || k > 8 || k == 7) return false;
    switch (kernel) {
        case TWS_KERNEL_TILE_128x128: shape_of<2, 8, 16>(k, out); return true;
        case TWS_KERNEL_TILE_128x64: shape_of<2, 8, 8>(k, out); return true;
        case TWS_KERNEL_TILE_256x64: shape_of<4, 4, 16>(k, out); return true;
        case TWS_KERNEL_TILE_64x64: shape_of<1, 8, 8>(k, out); return true;
        case TWS_KERNEL_TILE_64x64_16W: shape_of<1, 4, 16>(k, out); return true;
        case TWS_KERNEL_TILE_64x48_16W: shape_of<1, 3, 16>(k, out); return true;
        default: return false;
    }
}

template <class Args>
static hipError_t launch_tile_any(int kernel, int k, int mode, const Args& args, int blocks,
                                  const DryMaps& dry, hipStream_t s) {
    if (blocks <= 0) return hipSuccess;
    switch (kernel) {
        case TWS_KERNEL_TILE_128x128: return launch_tile_k<2, 8, 16>(k, mode, args, blocks, dry, s);
        case TWS_KERNEL_TILE_128x64: return launch_tile_k<2, 8, 8>(k, mode, args, blocks, dry, s);
        case TWS_KERNEL_TILE_256x64: return launch_tile_k<4, 4, 16>(k, mode, args, blocks, dry, s);
        case TWS_KERNEL_TILE_64x64: return launch_tile_k<1, 8, 8>(k, mode, args, blocks, dry, s);
        case TWS_KERNEL_TILE_64x64_16W: return launch_tile_k<1, 4, 16>(k, mode, args, blocks, dry, s);
        case TWS_KERNEL_TILE_64x48_16W: return launch_tile_k<1, 3, 16>(k, mode, args, blocks, dry, s);
        default: return hipErrorInvalidValue;
    }
}

int kernel_mode(const GridDesc& g) {
    if (truncated(g)) return kModeTruncated;
    if (g.boundary != TWS_BOUNDARY_CLOSED) return kModeGeneral;
    return g.rain_on != 0 ? kModeRain : kModePlain;
}

hipError_t launch_tile_batch(int kernel, int k, int mode, const GridDesc* grids_dev,
                             const int* hdr_dev, int blocks, int launch_idx, const DryMaps& dry,
                             hipStream_t s) {
    return launch_tile_any(kernel, k, mode, GridTable{grids_dev, hdr_dev, launch_idx}, blocks, dry, s);
}

hipError_t launch_tile_single(int kernel, int k, const GridDesc& g, const DryMaps& dry,
                              hipStream_t s) {
    return launch_tile_any(kernel, k, kernel_mode(g), OneGrid{tile_grid(g)},
                           g.tiles_x * g.tiles_y, dry, s);
}

hipError_t launch_twopass(const GridDesc* /*g_dev*/, const GridDesc& g, int parity,
                          hipStream_t s) {
    if (g.rain_on && g.brush_w > 0 && g.brush_h > 0)
        hipLaunchKernelGGL(k_brush, cell_grid(g), dim3(256), 0, s, g, parity, g.rain_cx, g.rain_cy,
                           g.rain_I, g.rain_R2);
    hipLaunchKernelGGL(k_flux_twopass, cell_grid(g), dim3(256), 0, s, g, parity);
    hipLaunchKernelGGL(k_apply_twopass, cell_grid(g), dim3(256), 0, s, g, parity);
    return hipGetLastError();
}

hipError_t launch_brush(const GridDesc& g, int parity, float cx, float cy, float I, float R2,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_brush, cell_grid(g), dim3(256), 0, s, g, parity, cx, cy, I, R2);
    return hipGetLastError();
}

hipError_t launch_velocity(const GridDesc& g, int parity, float* v2, hipStream_t s) {
    hipLaunchKernelGGL(k_velocity, cell_grid(g), dim3(256), 0, s, g, parity, v2);
    return hipGetLastError();
}

hipError_t launch_interleave(const GridDesc& g, int parity, float* staging4, hipStream_t s) {
    hipLaunchKernelGGL(k_interleave, cell_grid(g), dim3(256), 0, s, g, parity, staging4);
    return hipGetLastError();
}

hipError_t launch_deinterleave(const GridDesc& g, int parity, const float* staging4,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_deinterleave, cell_grid(g), dim3(256), 0, s, g, parity, staging4);
    return hipGetLastError();
}

hipError_t launch_ref_unpack(const GridDesc& g, int parity, const float* terrain_rgba,
                             const float* flow_rgba, float* b_out, hipStream_t s) {
    hipLaunchKernelGGL(k_ref_unpack, cell_grid(g), dim3(256), 0, s, g, parity, terrain_rgba,
                       flow_rgba, b_out);
    return hipGetLastError();
}

hipError_t launch_ref_pack(const GridDesc& g, int parity, float gb_fill, float* terrain_rgba,
                           float* flow_rgba, uint16_t* flowmap, hipStream_t s) {
    hipLaunchKernelGGL(k_ref_pack, cell_grid(g), dim3(256), 0, s, g, parity, gb_fill, terrain_rgba,
                       flow_rgba, flowmap);
    return hipGetLastError();
}

hipError_t launch_volume_partials(const GridDesc& g, int parity, double* partials, int nparts,
                                  hipStream_t s) {
    hipLaunchKernelGGL(k_volume, dim3(nparts), dim3(256), 0, s, g, parity, partials, nparts);
    return hipGetLastError();
}

hipError_t launch_zero_fill(float* p, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_zero_fill, dim3((unsigned)blocks), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

hipError_t launch_fbm(float* b, const GridDesc& g, uint64_t seed, int octaves, int base,
                      double persistence, double scale, hipStream_t s) {
    hipLaunchKernelGGL(k_fbm, cell_grid(g), dim3(256), 0, s, b, g.pitch, g.W, g.H, seed, octaves,
                       base, persistence, scale);
    return hipGetLastError();
}

hipError_t launch_init_water(const GridDesc& g, int parity, float depth, int x0, int y0, int x1,
                             int y1, float rect_depth, hipStream_t s) {
    hipLaunchKernelGGL(k_init_water, cell_grid(g), dim3(256), 0, s, g, parity, depth, x0, y0, x1,
                       y1, rect_depth);
    return hipGetLastError();
}

hipError_t launch_check_finite(const GridDesc& g, int parity, hipStream_t s) {
    hipLaunchKernelGGL(k_check_finite, cell_grid(g), dim3(256), 0, s, g, parity);
    return hipGetLastError();
}

// Launch shapes of the copy: (loads in flight per lane, non-temporal,
// work groups of 256 per CU).
struct CopyShape {
    int unroll;
    bool nt;
    int groups_per_cu;
};
static const CopyShape kCopyShapes[] = {
    {1, false, 64},  // one load per lane and iteration
    {4, false, 8}, {4, true, 8}, {8, true, 4}, {8, true, 8}, {4, true, 16}, {8, false, 8},
};
int stream_copy_shapes() { return (int)(sizeof(kCopyShapes) / sizeof(kCopyShapes[0])); }

hipError_t launch_stream_copy(const void* src, void* dst, int64_t bytes, int shape,
                              hipStream_t s) {
    if (shape < 0 || shape >= stream_copy_shapes()) return hipErrorInvalidValue;
    const CopyShape& c = kCopyShapes[shape];
    const int64_t n = bytes / 16;
    if (n < 1) return hipSuccess;
    int64_t blocks = (n + 256LL * c.unroll - 1) / (256LL * c.unroll);
    blocks = std::min<int64_t>(blocks, 256LL * c.groups_per_cu);
    const vf4* sv = static_cast<const vf4*>(src);
    vf4* dv = static_cast<vf4*>(dst);
    const dim3 grid((unsigned)blocks), block(256);
    if (c.unroll == 1) hipLaunchKernelGGL((k_stream_copy<1, false>), grid, block, 0, s, sv, dv, n);
    else if (c.unroll == 4 && !c.nt) hipLaunchKernelGGL((k_stream_copy<4, false>), grid, block, 0, s, sv, dv, n);
    else if (c.unroll == 4) hipLaunchKernelGGL((k_stream_copy<4, true>), grid, block, 0, s, sv, dv, n);
    else if (!c.nt) hipLaunchKernelGGL((k_stream_copy<8, false>), grid, block, 0, s, sv, dv, n);
    else hipLaunchKernelGGL((k_stream_copy<8, true>), grid, block, 0, s, sv, dv, n);
    return hipGetLastError();
}

hipError_t launch_lane_shift_probe(int* out128, hipStream_t s) {
    hipLaunchKernelGGL(k_lane_shift_probe, dim3(1), dim3(64), 0, s, out128);
    return hipGetLastError();
}

}  // namespace tws
