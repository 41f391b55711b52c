// tws_tune.cpp -- launch configuration of the fused step kernel: the default
// table and the measuring autotuner.
//
// choose_launch() maps a grid size to (kernel variant, steps per launch).
// Grids up to 2176^2, and larger ones on other edges than closed walls, take
// the tile launch that a measured table of launch times by rounds of tiles
// makes the fastest (tile_launch); grids above 2176^2 in closed walls the
// streaming kernel at k = 6.
// tws_autotune() times every candidate (the tile variants and the streaming
// kernel, each at k = 2..6 and 8) on scratch grids of the requested shapes
// advanced as one batch and returns the winner; only tws_tune_record() enters a launch into
// the per-size-class table (log2 of the cell count) that choose_launch()
// consults first, so tuning a batch never changes what a later plain grid
// of the process runs.

#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <map>
#include <mutex>
#include <vector>

#include "tws.h"
#include "tws_runtime.hpp"

namespace tws {

static std::mutex g_tune_mu;
static std::map<int, std::pair<int, int>> g_tuned;  // size class -> (kernel, k)

static int size_class(int64_t cells) {
    int c = 0;
    while (cells > 1) { cells >>= 1; ++c; }
    return c;
}

// What a tile launch takes, by rounds of tiles.  A launch lasts as long as the
// compute units (256) need for their rounds of work groups: a CU that holds two
// runs both at half speed, so the time is a function of tiles / 256, rounded
// up, and hardly of anything else; within the first round it grows a little
// with every tile.  MI355X, us per launch of k steps on square grids of
// 128^2..2304^2 (0.5 m sheet, closed walls; a rain disc adds 1-3%): few tiles,
// then 256, 512, ... 2048 tiles.
struct TileCost {
    int kernel, k;
    float few, rounds[8];
};
static const TileCost kTileCosts[] = {
    {TWS_KERNEL_TILE_64x48_16W, 4, 9.3f, {12.7f, 17.9f, 21.4f, 25.4f, 30.6f, 35.3f, 39.9f, 44.4f}},
    {TWS_KERNEL_TILE_64x48_16W, 5, 10.2f, {12.8f, 19.2f, 24.0f, 27.5f, 33.1f, 38.5f, 43.8f, 48.9f}},
    {TWS_KERNEL_TILE_64x48_16W, 6, 11.2f, {13.3f, 19.6f, 26.2f, 30.1f, 35.5f, 41.3f, 47.5f, 53.2f}},
    {TWS_KERNEL_TILE_64x48_16W, 8, 12.6f, {14.1f, 20.7f, 29.0f, 35.7f, 42.0f, 48.2f, 54.3f, 61.4f}},
    {TWS_KERNEL_TILE_64x64_16W, 4, 11.2f, {16.4f, 20.3f, 26.0f, 32.2f, 38.6f, 44.5f, 50.1f, 55.9f}},
    {TWS_KERNEL_TILE_64x64_16W, 5, 12.5f, {16.9f, 22.9f, 28.3f, 34.9f, 42.2f, 49.0f, 56.1f, 62.5f}},
    {TWS_KERNEL_TILE_64x64_16W, 6, 13.7f, {17.5f, 25.0f, 31.0f, 38.4f, 46.1f, 53.6f, 62.0f, 69.5f}},
    {TWS_KERNEL_TILE_64x64_16W, 8, 15.9f, {18.4f, 27.8f, 36.6f, 43.8f, 52.9f, 61.5f, 71.2f, 80.6f}},
    {TWS_KERNEL_TILE_64x64, 4, 13.0f, {18.7f, 22.0f, 27.0f, 32.8f, 40.5f, 46.2f, 51.0f, 56.0f}},
    {TWS_KERNEL_TILE_64x64, 5, 14.5f, {19.0f, 24.8f, 29.8f, 36.3f, 42.9f, 51.1f, 57.2f, 63.5f}},
    {TWS_KERNEL_TILE_64x64, 6, 16.1f, {19.7f, 27.0f, 32.3f, 38.2f, 45.1f, 51.8f, 60.8f, 67.7f}},
    {TWS_KERNEL_TILE_128x64, 5, 22.8f, {26.4f, 38.6f, 53.5f, 69.2f, 81.5f, 94.0f, 107.0f, 120.0f}},
    {TWS_KERNEL_TILE_128x64, 6, 25.8f, {28.9f, 43.0f, 59.6f, 75.4f, 91.6f, 107.0f, 123.0f, 139.0f}},
};

static float launch_us(const TileCost& c, int64_t tiles) {
    const float r = (float)tiles / 256.0f;
    if (r <= 1.0f) return c.few + (c.rounds[0] - c.few) * r;
    if (r <= 8.0f) return c.rounds[(tiles + 255) / 256 - 1];
    return c.rounds[7] + (r - 8.0f) * 0.5f * (c.rounds[7] - c.rounds[5]);
}

void choose_launch(int width, int height, int* kernel, int* k) {
    const int64_t cells = (int64_t)width * height;
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        auto it = g_tuned.find(size_class(cells));
        if (it != g_tuned.end()) {
            *kernel = it->second.first;
            *k = it->second.second;
            return;
        }
    }
    // Above 2176^2 the streaming kernel at k = 6 leads (closed walls; other
    // boundaries step on tile_launch's choice).  MI355X, 0.5 m sheet on fBm
    // terrain in closed walls, cell-updates/s stream (k = 6) vs the tile
    // table: 2048^2 2.71e11 (k = 5: 2.89e11) vs 3.02e11, 2304^2 3.19e11
    // (k = 5: 3.22e11) vs 2.95e11, 2560^2 3.50e11 vs 3.15e11, 2816^2 3.70e11
    // vs 3.29e11, 3072^2 3.96e11 vs 3.40e11; 4096^2 4.42e11 vs 3.67e11, 8192^2
    // 4.61e11 vs 3.98e11 and 16384^2 5.3e11 vs 4.26e11 in other runs.
    if (cells > 2176 * 2176) {
        *kernel = TWS_KERNEL_STREAM_128;
        *k = 6;
        return;
    }
    tile_launch(width, height, kernel, k);
}

void tile_launch(int width, int height, int* kernel, int* k) {
    const int64_t cells = (int64_t)width * height;
    // Up to 1536^2 cells the launch that takes least per step by kTileCosts.
    // Against one launch per band of sizes, us per 96 steps: 640^2 with rain 292
    // vs 381, 864^2 with rain 413 vs 557, 960^2 428 vs 516, 1024^2 with rain 487
    // vs 520, 1152^2 with rain 568 vs 644, 1408^2 693 vs 768, 100 x 8000 450 vs
    // 517; 256^2 and 512^2 keep theirs.  Past 6 rounds the candidates come
    // within a few percent and memory has its say:
    //   <= 2304^2  64x64 tiles, 8 waves, k = 4: 2048^2 zero edge, us per 96
    //              steps, 1343 vs 1428 for 64x64 over 16 waves, k = 5, with a
    //              lake in closed walls 1314 vs 1382; 1800^2 zero edge 1086 vs
    //              1150 for 128x64, k = 5
    //   <= 3072^2  64x64, k = 5 (zero edge, all wet, us per 96 steps): 2500^2
    //              1718 vs 1950 for 128x64, k = 5 and 1780 at k = 4; 3001 x 2777
    //              2387 either way, and its smaller tiles pass over more once
    //              the ground dries
    //   <= 4096^2  128x64, k = 5: 4096^2 4300 us vs 4527 for 64x64, k = 5
    //   larger     128x64, k = 4: the 16384^2 dam-break 4.30e11 vs 4.10e11 at
    //              k = 5 (on an all-wet 16384^2 sheet k = 5 leads by 4%).
    if (cells <= 1536 * 1536) {
        float best = 0.0f;
        for (const TileCost& c : kTileCosts) {
            TileShape sh{};
            if (!tile_shape(c.kernel, c.k, &sh)) continue;
            const int64_t tiles = (int64_t)((width + sh.ox - 1) / sh.ox) * ((height + sh.oy - 1) / sh.oy);
            const float us = launch_us(c, tiles) / (float)c.k;
            if (best == 0.0f || us < best) {
                best = us;
                *kernel = c.kernel;
                *k = c.k;
            }
        }
    } else if (cells <= 2304 * 2304) {
        *kernel = TWS_KERNEL_TILE_64x64;
        *k = 4;
    } else if (cells <= 3072 * 3072) {
        *kernel = TWS_KERNEL_TILE_64x64;
        *k = 5;
    } else if (cells <= 4096 * 4096) {
        *kernel = TWS_KERNEL_TILE_128x64;
        *k = 5;
    } else {
        *kernel = TWS_KERNEL_TILE_128x64;
        *k = 4;
    }
}

// Tile order of the step kernel for a grid's default launch: groups of
// tile columns walked row by row (tws_set_tile_order).  MI355X, 4096^2 plain
// sheet at 128x64 / k = 5 (38 tile columns): 3.81e11 cell-updates/s with
// groups of 20 against 3.74e11 with 16, 3.78e11 with 24, 3.73e11 row-major;
// other sizes keep 16 (at 16384^2 and k = 4, widths of 21-37 and 16 came within
// 2% of each other and 25 lost 3%).
int default_tile_group(int width, int height, int kernel, int k) {
    const int64_t cells = (int64_t)width * height;
    if (kernel == TWS_KERNEL_STREAM_128) tile_launch(width, height, &kernel, &k);
    if (kernel == TWS_KERNEL_TILE_128x64 && k == 5 && cells > 2048 * 2048 && cells <= 4096 * 4096)
        return 20;
    return 16;
}

}  // namespace tws

using namespace tws;

extern "C" {

int tws_autotune(const int32_t* widths, const int32_t* heights, int32_t n, int32_t steps,
                 tws_tune_entry* best, tws_tune_entry* results, int32_t capacity,
                 int32_t* count) {
    if (!widths || !heights || n <= 0 || steps <= 0 || !best)
        return fail(TWS_ERR_INVALID, "tws_autotune: invalid argument");
    int64_t bytes = 0, cells = 0;
    for (int i = 0; i < n; ++i) {
        if (widths[i] <= 0 || heights[i] <= 0)
            return fail(TWS_ERR_INVALID, "tws_autotune: invalid shape %d", i);
        bytes += tws_grid_footprint(widths[i], heights[i]);
        cells += (int64_t)widths[i] * heights[i];
    }
    tws_params p{};
    int rc = tws_params_physical(0.02f, 9.81f, 1.0f, 1.0f, 0.995f, TWS_BOUNDARY_CLOSED, &p);
    if (rc != TWS_OK) return rc;
    tws_batch* b = nullptr;
    rc = tws_batch_create(n, bytes, nullptr, &b);
    if (rc != TWS_OK) return rc;
    // synthetic wet state: fBm terrain 0..100 m under a 0.5 m sheet, and a
    // rain disc (r = 16) at the centre as in the batched and served
    // workloads, so the kernel timed is the one with the rain source
    std::vector<float> terrain, depth;
    for (int i = 0; i < n && rc == TWS_OK; ++i) {
        int32_t id = -1;
        rc = tws_batch_add(b, widths[i], heights[i], &p, &id);
        if (rc != TWS_OK) break;
        const size_t c = (size_t)widths[i] * heights[i];
        try {
            terrain.resize(c);
            depth.assign(c, 0.5f);
        } catch (...) {
            rc = fail(TWS_ERR_NOMEM, "tws_autotune: host allocation failed");
            break;
        }
        rc = tws_generate_fbm_terrain(widths[i], heights[i], 1000u + (uint64_t)i, 6, 4, 0.43f,
                                      100.0f, terrain.data());
        if (rc == TWS_OK) rc = tws_batch_upload(b, id, terrain.data(), depth.data(), nullptr);
        if (rc == TWS_OK)
            rc = tws_batch_set_rain(b, id, 0.5f * widths[i], 0.5f * heights[i], 1e-3f, 256.0f);
    }
    static const int kernels[] = {TWS_KERNEL_TILE_128x64,    TWS_KERNEL_TILE_128x128,
                                  TWS_KERNEL_TILE_256x64,    TWS_KERNEL_TILE_64x64,
                                  TWS_KERNEL_TILE_64x64_16W, TWS_KERNEL_TILE_64x48_16W,
                                  TWS_KERNEL_STREAM_128};
    static const int ks[] = {2, 3, 4, 5, 6, 8};
    tws_tune_entry top{0, 0, 0.0};
    int m = 0;
    for (int kern : kernels) {
        for (int kk : ks) {
            if (rc != TWS_OK) break;
            rc = tws_batch_set_launch(b, kern, kk);
            // warm with the same step count: the timed run then replays the
            // captured launch sequence instead of capturing one
            if (rc == TWS_OK) rc = tws_batch_step(b, steps);
            if (rc == TWS_OK) rc = tws_batch_sync(b);
            const auto t0 = std::chrono::steady_clock::now();
            if (rc == TWS_OK) rc = tws_batch_step(b, steps);
            if (rc == TWS_OK) rc = tws_batch_sync(b);
            const double sec =
                std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            if (rc != TWS_OK) break;
            const tws_tune_entry e{kern, kk, (double)cells * steps / sec};
            if (results && m < capacity) results[m] = e;
            ++m;
            if (e.cell_updates_per_s > top.cell_updates_per_s) top = e;
        }
    }
    tws_batch_destroy(b);
    if (rc != TWS_OK) return rc;
    if (count) *count = m;
    *best = top;
    return TWS_OK;
}

int tws_tune_record(int32_t width, int32_t height, int32_t kernel, int32_t k) {
    if (width <= 0 || height <= 0)
        return fail(TWS_ERR_INVALID, "tws_tune_record: invalid size %d x %d", width, height);
    TileShape sh{};
    int ox = 0;
    if (!(kernel == TWS_KERNEL_STREAM_128 ? k >= 2 && stream_shape(k, &ox) : tile_shape(kernel, k, &sh)))
        return fail(TWS_ERR_INVALID, "tws_tune_record: unknown kernel %d or k %d", kernel, k);
    std::lock_guard<std::mutex> lk(g_tune_mu);
    try {
        g_tuned[size_class((int64_t)width * height)] = {kernel, k};
    } catch (...) {
        return fail(TWS_ERR_NOMEM, "tws_tune_record: host allocation failed");
    }
    return TWS_OK;
}

int tws_tune_forget(void) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned.clear();
    return TWS_OK;
}

}  // extern "C"
