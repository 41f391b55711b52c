// tws_active.hip -- which part of a grid the streaming step kernel works on.
//
// A cell that holds neither water nor flux keeps both at +0 through a step
// unless a neighbour drains into it, so dry ground more than n cells from
// anything wet is dry after n steps too.  In a dam-break, under rain on dry
// terrain and in a sheet that has drained into the basins most of a grid is
// such ground.  Within one run of launches (nothing outlives the call), every
// few launches
//   k_survey  looks at the current state in bands of kBand rows by one strip
//             (the streaming kernel's output columns) and notes which hold
//             anything but dry cells; it zeroes the other buffer set under
//             the dry ones, so that a band left alone is right in both sets;
//   k_plan    takes the bands within reach of a wet band until the next
//             survey (the active ones), and cuts their rows into segments of
//             one length, as many as the device runs at once.
// The launches until the next survey step these segments and nothing else.
//
// k_survey calls a band dry only where that holds to the bit: see
// regular_height (tws_kernel_util.hpp).

#include <hip/hip_runtime.h>

#include <algorithm>

#include "tws.h"
#include "tws_internal.hpp"
#include "tws_kernel_util.hpp"

namespace tws {

namespace {

constexpr int kBand = kActiveBand;    // rows per band
constexpr int kBandsPerWord = 64;     // bands per word of a mask
constexpr int kSurveyWaves = 16;      // wavefronts of a survey work group, a band each
constexpr int kSurveyParts = kBandsPerWord / kSurveyWaves;  // work groups per word
constexpr int kPlanThreads = 1024;
constexpr int kPlanWords = 6144;      // words k_plan can plan (in LDS)
constexpr int kReachBands = kActiveReach / kBand;
// Rounds (a survey and its plan) until a state found all wet is looked at
// again.  MI355X, 100 steps of the wet 4096^2 sheet (3.9 ms, 4 rounds of k = 6):
// 2.0% for the rounds when each looks, 1.0% when only the first does; 1000 steps
// in one call 34.5 ms looking every 4 rounds, 34.3 every 8.
constexpr int kFullRounds = 8;
constexpr int kMinRows = 16;          // shortest segment worth a wavefront

// Words of a grid's masks: any | left | right | active, strips x words each.
__device__ __forceinline__ uint64_t* mask_of(const GridDesc& g, int strips, int which) {
    return g.bands + (int64_t)which * strips * g.band_words;
}

// The grid that flattened index `i` falls in (grids ordered by `first`).
template <class First>
__device__ __forceinline__ int find_grid(int n, int i, First first) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first(mid) <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
}

}  // namespace

// A wavefront per band, 2 columns per lane; a work group writes a quarter word
// of each mask.  Bound by memory where the ground is dry for the first time (20
// B per cell read, 20 B written, and the heights) and by latency elsewhere: a
// band whose first four rows of depth are wet at both sides is read no
// further, and a band that was dry at the last survey too is not written.
template <bool BATCH>
__global__ void __launch_bounds__(kSurveyWaves * kWave)
__attribute__((amdgpu_waves_per_eu(4, 4)))  // registers for the loads in flight
k_survey(GridDesc g1, const GridDesc* __restrict__ grids, const int* __restrict__ hdr,
         int launch_idx, int strips1, int parity1, int k, int out_cols, int parts, int round,
         const int* __restrict__ count) {
    // After a round that found nearly all of it active, every row is stepped
    // until a round looks again, at all bands: their marks are out of date.
    const bool first = round == 0 || *count < 0;
    if (round != 0 && first && round % kFullRounds != 0) return;
    __shared__ int s_wet[kSurveyWaves];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    GridDesc g;
    int strips = strips1, parity = parity1;
    if constexpr (!BATCH) g = g1;
    // Contiguous runs of parts per XCD, neighbouring strips after each other: a
    // strip's rows share cache lines with the next strip's.
    const int nb = gridDim.x, xcd = blockIdx.x & 7, q8 = nb >> 3, rmd = nb & 7;
    int item = xcd * q8 + min(xcd, rmd) + (blockIdx.x >> 3);
    if constexpr (BATCH) {  // a part per work group
        const GridDesc* table = grids + hdr[2];
        const int n = hdr[0];
        if (n <= 0) return;
        const int i = find_grid(n, item / kSurveyParts, [&](int m) { return table[m].word_begin; });
        g = table[__builtin_amdgcn_readfirstlane(i)];
        if (g.steps < (launch_idx + 1) * k) return;  // not in this launch: its state is elsewhere
        item -= g.word_begin * kSurveyParts;
        strips = g.tiles_x;
        parity = (g.parity0 + launch_idx) & 1;
        parts = strips * g.band_words * kSurveyParts;
    }
    for (; item < parts; item += BATCH ? parts : nb) {
    const int word = item / (strips * kSurveyParts), in_word = item - word * strips * kSurveyParts;
    const int part = in_word / strips, strip = in_word - part * strips;
    const int64_t at = (int64_t)strip * g.band_words + word;
    // a part with no active band keeps its masks: nothing there was or is wet
    if (!first && reinterpret_cast<const uint16_t*>(mask_of(g, strips, 3) + at)[part] == 0) continue;
    const int W = g.W, H = g.H;
    const int band = word * kBandsPerWord + part * kSurveyWaves + wave, y0 = band * kBand;
    const int x = strip * out_cols + lane * 2;  // even: both columns lie in the row's pitch
    const bool own = lane * 2 < out_cols && x < W;
    const bool two = x + 1 < W;
    // what the neighbouring strips need to know: anything wet within reach
    const uint64_t left_lanes = strip > 0 ? ~0ull >> (64 - kActiveReach / 2) : 0;
    const uint64_t right_lanes = strip + 1 < strips ? ~0ull << ((out_cols - kActiveReach) / 2) : 0;
    const int bit = part * kSurveyWaves + wave;
    const bool look = y0 < H && (first || ((mask_of(g, strips, 3)[at] >> bit) & 1));
    const bool was_dry = !first && !((mask_of(g, strips, 0)[at] >> bit) & 1);
    const float* in[5] = {parity ? g.d[1] : g.d[0], parity ? g.f[1][0] : g.f[0][0],
                          parity ? g.f[1][1] : g.f[0][1], parity ? g.f[1][2] : g.f[0][2],
                          parity ? g.f[1][3] : g.f[0][3]};
    float* out[5] = {parity ? g.d[0] : g.d[1], parity ? g.f[0][0] : g.f[1][0],
                     parity ? g.f[0][1] : g.f[1][1], parity ? g.f[0][2] : g.f[1][2],
                     parity ? g.f[0][3] : g.f[1][3]};
    const int xc = own ? x : 0;
    auto bits = [&](const float* plane, int y) {  // rows past the end read the last row again
        const vf2 v = *reinterpret_cast<const gfloat2*>(gptr(plane) + (int64_t)min(y, H - 1) * g.pitch + xc);
        return __float_as_uint(v.x) | (two ? __float_as_uint(v.y) : 0u);
    };
    uint64_t wet = 0;
    if (look) {
        uint32_t u = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) u |= bits(in[0], y0 + r);
        wet = __ballot(own && u != 0);
        const bool sides = (!left_lanes || (wet & left_lanes)) && (!right_lanes || (wet & right_lanes));
        if (!wet || !sides) {
#pragma unroll
            for (int half = 0; half < kBand; half += kBand / 2) {
                uint32_t v[5] = {0, 0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < kBand / 2; ++r)
#pragma unroll
                    for (int p = 0; p < 5; ++p) v[p] |= bits(in[p], y0 + half + r);
                u |= v[0] | v[1] | v[2] | v[3] | v[4];
            }
            wet = __ballot(own && u != 0);
        }
        if (!wet && !was_dry) {
            // heights of the band and one cell around it
            bool ok = g.dry_ok != 0;
            const int xb = min(max(x - 2, 0), (int)g.pitch - 2);
            if (lane * 2 < out_cols + 4) {
                bool good[2] = {true, true};
#pragma unroll
                for (int r = -1; r <= kBand; ++r) {
                    const int y = min(max(y0 + r, 0), H - 1);
                    const vf2 b = *reinterpret_cast<const gfloat2*>(gptr(g.b) + (int64_t)y * g.pitch + xb);
                    good[0] = good[0] && regular_height(b.x);
                    good[1] = good[1] && regular_height(b.y);
                }
                ok = ok && (xb >= W || good[0]) && (xb + 1 >= W || good[1]);
            }
            if (__ballot(!ok) != 0) {
                wet = ~0ull;
            } else if (own) {
#pragma unroll
                for (int r = 0; r < kBand; ++r) {
                    if (y0 + r >= H) break;
                    const int64_t off = (int64_t)(y0 + r) * g.pitch + x;
#pragma unroll
                    for (int p = 0; p < 5; ++p)
                        *reinterpret_cast<gfloat2*>(gptr(out[p]) + off) = vf2{0.0f, 0.0f};
                }
            }
        }
    }
    if (lane == 0)
        s_wet[wave] = (wet ? 1 : 0) | (wet & left_lanes ? 2 : 0) | (wet & right_lanes ? 4 : 0);
    __syncthreads();
    if (threadIdx.x < 3) {
        uint32_t m = 0;
        for (int w = 0; w < kSurveyWaves; ++w) m |= (uint32_t)((s_wet[w] >> threadIdx.x) & 1) << w;
        reinterpret_cast<uint16_t*>(mask_of(g, strips, threadIdx.x) + at)[part] = (uint16_t)m;
    }
    __syncthreads();
    }
}

namespace {

// The bands of word w of a strip that are wet, that a neighbouring strip's
// water reaches, or that it rains on.
__device__ __forceinline__ uint64_t wet_word(const GridDesc& g, int strips, int strip, int w,
                                             int out_cols) {
    const int words = g.band_words;
    if (w < 0 || w >= words) return 0;
    const int64_t at = (int64_t)strip * words + w;
    uint64_t m = mask_of(g, strips, 0)[at];
    if (strip + 1 < strips) m |= mask_of(g, strips, 1)[at + words];
    if (strip > 0) m |= mask_of(g, strips, 2)[at - words];
    if (g.rain_on) {
        const int x = strip * out_cols;
        double top, bottom;
        if (brush_span(g, x - kActiveReach, x + out_cols - 1 + kActiveReach, top, bottom)) {
            const int lo = max((int)top / kBand - w * kBandsPerWord, 0);
            const int hi = min((int)bottom / kBand - w * kBandsPerWord, kBandsPerWord - 1);
            if (lo <= hi) m |= (~0ull << lo) & (~0ull >> (63 - hi));
        }
    }
    return m;
}

// The active bands of word w: those within kReachBands of a wet one, and
// single bands between active ones (a segment's ramp costs more than a band).
__device__ __forceinline__ uint64_t active_word(const GridDesc& g, int strips, int strip, int w,
                                                int out_cols) {
    const uint64_t prev = wet_word(g, strips, strip, w - 1, out_cols);
    const uint64_t cur = wet_word(g, strips, strip, w, out_cols);
    const uint64_t next = wet_word(g, strips, strip, w + 1, out_cols);
    uint64_t m = cur;
#pragma unroll
    for (int r = 1; r <= kReachBands; ++r)
        m |= cur << r | cur >> r | prev >> (64 - r) | next << (64 - r);
    m |= (m << 1) & (m >> 1);
    const int n = (g.H + kBand - 1) / kBand - w * kBandsPerWord;
    return n >= 64 ? m : m & ((1ull << n) - 1);
}

}  // namespace

// One work group plans the launches until the next survey: list[i] = {strip,
// first row, end row, grid}, *count entries, at most max_tasks; or *count = -1,
// the static plan, where that does not do or nearly all rows are active.
// Segments do not cross words (1024 rows).  Bound by the latency of a few
// dependent passes over the words, a thread each: making the active words, then
// cutting their runs of bands.
template <bool BATCH>
__global__ void __launch_bounds__(kPlanThreads)
k_plan(GridDesc g1, const GridDesc* __restrict__ grids, const int* __restrict__ hdr,
       int launch_idx, int strips1, int k, int out_cols, int slots, int max_rows, int max_tasks,
       int round, int4* __restrict__ list, int* __restrict__ count) {
    if (round % kFullRounds != 0 && *count < 0) return;  // as k_survey
    __shared__ uint64_t s_act[kPlanWords];
    __shared__ int s_rows, s_runs, s_all;
    __shared__ int s_wave[kPlanThreads / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const GridDesc* table = BATCH ? grids + hdr[2] : nullptr;
    const int n_grids = BATCH ? hdr[0] : 1;
    int words = 0;
    if constexpr (BATCH) {
        if (n_grids > 0) {
            const GridDesc& g = table[n_grids - 1];
            words = g.word_begin + g.tiles_x * g.band_words;
        }
    } else {
        words = strips1 * g1.band_words;
    }
    auto grid_at = [&](int i) {
        return BATCH ? find_grid(n_grids, i, [&](int m) { return table[m].word_begin; }) : 0;
    };
    auto grid_of = [&](int gi) -> const GridDesc& { return BATCH ? table[gi] : g1; };
    if (tid == 0) s_rows = s_runs = s_all = 0;
    __syncthreads();
    int rows = 0, runs = 0, all = 0;
    for (int i = tid; i < words; i += kPlanThreads) {
        const GridDesc& g = grid_of(grid_at(i));
        uint64_t m = 0;
        // grids that are not in this launch keep no masks current
        if (!BATCH || g.steps >= (launch_idx + 1) * k) {
            const int local = i - g.word_begin;
            const int strip = local / g.band_words, w = local - strip * g.band_words;
            const int strips = BATCH ? g.tiles_x : strips1;
            m = active_word(g, strips, strip, w, out_cols);
            mask_of(g, strips, 3)[local] = m;
            const int y0 = w * kBandsPerWord * kBand, n = min(g.H - y0, kBandsPerWord * kBand);
            all += n;
            rows += min(__popcll(m) * kBand, n);
            runs += __popcll(m & ~(m << 1));
        }
        if (i < kPlanWords) s_act[i] = m;
    }
    if (all) atomicAdd(&s_all, all);
    if (rows) atomicAdd(&s_rows, rows);
    if (runs) atomicAdd(&s_runs, runs);
    __syncthreads();
    // As many segments as fill the wavefront slots once, or a whole number of
    // times where a segment would run past max_rows.
    const int rounds = max(1, (s_rows / slots + max_rows - 1) / max_rows);
    const int free_slots = slots * rounds - s_runs;
    // Only where a wavefront sweeps an eighth less than in the static plan, the 4 k
    // rows of a segment's ramps counted: fragments of active rows take slots and
    // ramps of their own, and surveying them takes some 5% of the launches.
    // (4096^2 sheet with a tenth of it dry, 1000 steps: 35.3 ms listed, 33.3 static.)
    const int all_rounds = max(1, (s_all / slots + max_rows - 1) / max_rows);
    const int all_len = (s_all + slots * all_rounds - 1) / (slots * all_rounds);
    const int len = free_slots > 0 ? max(kMinRows, (s_rows + free_slots - 1) / free_slots) : 0;
    if (words > kPlanWords || free_slots <= 0 ||
        (int64_t)(len + 4 * k) * rounds * 8 > (int64_t)(all_len + 4 * k) * all_rounds * 7) {
        if (tid == 0) *count = -1;
        return;
    }
    // Calls run(first band, rows) for the runs of a word's bands; `below`: rows
    // of the grid from the word's first on.
    auto each_run = [](uint64_t m, int below, auto run) {
        while (m) {
            const int from = __builtin_ctzll(m);
            const uint64_t holes = ~(m >> from);
            const int n = holes ? __builtin_ctzll(holes) : 64;
            run(from, min(n * kBand, below - from * kBand));
            m = from + n < 64 ? m & (~0ull << (from + n)) : 0;
        }
    };
    // Chunk by chunk: a word's tasks counted, their places summed over the
    // group, the tasks written (while they fit).
    int base = 0;
    for (int first = 0; first < words; first += kPlanThreads) {
        const int i = first + tid;
        const uint64_t m = i < words ? s_act[i] : 0;
        int n = 0, gi = 0, strip = 0, y = 0, below = 0;
        if (m) {
            gi = grid_at(i);
            const GridDesc& g = grid_of(gi);
            const int local = i - g.word_begin;
            strip = local / g.band_words;
            y = (local - strip * g.band_words) * kBandsPerWord * kBand;
            below = g.H - y;
            each_run(m, below, [&](int, int rows) { n += (rows + len - 1) / len; });
        }
        int scan = n;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int v = __shfl_up(scan, d);
            if (lane >= d) scan += v;
        }
        if (lane == kWave - 1) s_wave[wave] = scan;
        __syncthreads();
        int at = base + scan - n, sum = 0;
        for (int w = 0; w < kPlanThreads / kWave; ++w) {
            if (w < wave) at += s_wave[w];
            sum += s_wave[w];
        }
        __syncthreads();
        base += sum;
        if (at + n > max_tasks) continue;
        each_run(m, below, [&](int from, int rows) {
            const int q = (rows + len - 1) / len, part = rows / q;
            const int longer = rows - part * q;  // the first ones take a row more
            int y0 = y + from * kBand;
            for (int j = 0; j < q; ++j) {
                const int end = y0 + part + (j < longer ? 1 : 0);
                list[at++] = make_int4(strip, y0, end, gi);
                y0 = end;
            }
        });
    }
    if (tid == 0) *count = base <= max_tasks ? base : -1;
}

int64_t active_band_words(int H) {
    return ((H + kBand - 1) / kBand + kBandsPerWord - 1) / kBandsPerWord;
}

hipError_t launch_active(const ActiveRun& a, int parity, int launch_idx, int round,
                         hipStream_t s) {
    int out_cols = 0;
    if (!stream_shape(a.k, &out_cols) || !a.list || !a.count || a.survey_words <= 0)
        return hipErrorInvalidValue;
    const GridDesc g1 = a.grid ? *a.grid : GridDesc{};
    // every part in one go at first; later most parts have no active band
    const int parts = a.survey_words * kSurveyParts;
    const dim3 survey(round == 0 || !a.grid ? parts : std::min(parts, 1024)), waves(kSurveyWaves * kWave);
    const dim3 one(1), plan(kPlanThreads);
    if (a.grid) {
        hipLaunchKernelGGL((k_survey<false>), survey, waves, 0, s, g1, a.grids, a.hdr, launch_idx,
                           a.plan.strips, parity, a.k, out_cols, parts, round, a.count);
        hipLaunchKernelGGL((k_plan<false>), one, plan, 0, s, g1, a.grids, a.hdr, launch_idx,
                           a.plan.strips, a.k, out_cols, a.slots, kStreamSegRows, a.max_tasks,
                           round, a.list, a.count);
    } else {
        hipLaunchKernelGGL((k_survey<true>), survey, waves, 0, s, g1, a.grids, a.hdr, launch_idx,
                           0, 0, a.k, out_cols, parts, round, a.count);
        hipLaunchKernelGGL((k_plan<true>), one, plan, 0, s, g1, a.grids, a.hdr, launch_idx, 0,
                           a.k, out_cols, a.slots, kStreamSegRows, a.max_tasks, round, a.list,
                           a.count);
    }
    return hipGetLastError();
}

}  // namespace tws
