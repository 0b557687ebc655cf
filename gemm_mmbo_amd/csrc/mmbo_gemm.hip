// C ABI of the gfx950 GEMM library: argument checking, tile-config table, per-shape selection,
// split-K workspace and kernel dispatch.  The reference's counterpart is the header-inline host
// layer src/gemm/gemm.h (front-ends), src/gemm/constants.h (tables) and src/gemm/driver.h (launch).
#include "../../include/mmbo_gemm.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "configs.hpp"
#include "gemm_common.hpp"
#include "gemm_staged.hpp"
#include "gemm_wave.hpp"
#include "launch.hpp"
#include "tuned_table.hpp"

namespace mmbo {

namespace {

// Config ids (configs.hpp): [0, kStagedConfigs) are the staged kernel's (tile, split) pairs, then the ring kernel's
// (ring tile, split) pairs, then the x16 kernel's, then (fp32) the bf16 planes kernel's.  A ring config applies when m, n are multiples of its tile, k splits
// into whole slices and A, B are 16-byte aligned; otherwise the call is refused with MMBO_ERR_INVALID_CONFIG.
struct ConfigRef {
    bool ring;      // a direct-to-LDS kernel (ring or x16)
    int tile;
    int split;
    bool x16;
    bool planes;    // (neither ring nor x16)
};
inline ConfigRef config_ref(int id)
{
    if (id >= kPlanesBase) return {false, (id - kPlanesBase) % kPlanesIdTiles, kSplits[(id - kPlanesBase) / kPlanesIdTiles], false, true};
    if (id >= kX16Base) return {true, (id - kX16Base) % NUM_X16_TILES, kSplits[(id - kX16Base) / NUM_X16_TILES], true, false};
    if (id < kStagedConfigs) return {false, id % NUM_TILES, kSplits[id / NUM_TILES], false, false};
    id -= kStagedConfigs;
    return {true, id % NUM_RING_TILES, kSplits[id / NUM_RING_TILES], false, false};
}
inline bool valid_dtype(int dtype) { return dtype == MMBO_F32 || dtype == MMBO_F16 || dtype == MMBO_F64; }

// Does the ring (x16 = false) or x16 config (tile, split) take this shape?  Ring: m, n whole tiles, k whole slices, the
// same number for every split; A and B 16-byte aligned (checked at the call).  x16: any shape and alignment (its loads
// repeat or shift the last rows of an edge tile, its edge tiles store under guards, a partial last slice of k is
// zero-filled; the splits take equal runs of whole slices and the last one what is left, fewer splits than asked for
// when k is short) -- except a memory-contiguous m (transA = N) or n (transB = T) shorter than one 16-byte load.
inline bool ring_shape_ok(int dtype, int tile, int split, int transA, int transB, size_t m, size_t n, size_t k, bool x16)
{
    if (k == 0) return false;
    if (x16) {
        const size_t per16 = dtype == MMBO_F32 ? 4 : 8;
        return (transA || m >= per16) && (!transB || n >= per16);
    }
    const RingRow &r = kRingTiles[tile];
    const size_t bk = (size_t)ring_bk(dtype);
    if (m % r.bm || n % r.bn || k % bk) return false;
    return (k / bk) % (size_t)split == 0;
}

// ... the kernel on bf16 planes?  Any, except a memory-contiguous dimension shorter than one 16-byte load.
inline bool planes_shape_ok(int transA, int transB, size_t m, size_t n, size_t k) { return k >= 4 && (transA || m >= 4) && (!transB || n >= 4); }

thread_local int g_last_hip_error = 0;

int hip_fail(hipError_t e)
{
    g_last_hip_error = (int)e;
    return MMBO_ERR_HIP;
}

// ---- split-K workspace ------------------------------------------------------------------------
// A workspace holds the partial sums of one GEMM with GlobalSplitU > 1: [split][batch][n][m] fp32.
constexpr int kMaxDevices = 64;

// Library-owned workspaces: one per (device, stream), so GEMMs on different streams never share partial sums, grown on
// demand, at most kMaxWsSlots per device (the reference's launcher never frees what it loads, src/gemm/driver.h:41; this
// table is bounded instead).
//   - Each device has its own table and table lock, held only to look a slot up, add one or take one out.
//   - Each slot has its own lock, held by a call from the lookup until both launches that use the buffer (the GEMM and
//     the reduction) are queued: two host threads on one stream cannot interleave their launches, and growing a buffer
//     (wait for that stream, free, allocate) stalls only callers of that same stream.
//   - A buffer is never smaller than kWaveSumsBytes, what the split-by-wavefront kernel's splits take at most.
//   - A new stream that finds the table full retires the least recently used slot nobody holds: the table lock is given
//     up, the device is synchronised (the slot's stream may no longer exist, so it cannot be waited for by handle) and
//     the buffer freed.  mmbo_release_stream_workspace retires one stream's slot at the caller's request.
constexpr size_t kMaxWsSlots = 8;
// (work-groups of that kernel, splits included, that the automatic pick takes at most) x (sums of its largest tile)
constexpr size_t kMaxSplitWaveGroups = 1024;
constexpr size_t kWaveSumsBytes = kMaxSplitWaveGroups * 32 * 64 * sizeof(float);
constexpr bool wave_sums_fit(int i = 0) { return i == NUM_WAVE_TILES || (kMaxSplitWaveGroups * kWaveTiles[i].bm * kWaveTiles[i].bn * sizeof(float) <= kWaveSumsBytes && wave_sums_fit(i + 1)); }
static_assert(wave_sums_fit(), "the partial sums of the largest tile");
struct WsSlot {
    hipStream_t stream = nullptr;
    char *base = nullptr;
    size_t bytes = 0;
    unsigned long long last_use = 0;
    bool dead = false;          // taken out of the table; whoever still holds a reference looks the stream up again
    std::mutex use;
};
struct WsTable {
    std::mutex lock;
    std::vector<std::shared_ptr<WsSlot>> slots;
    unsigned long long clock = 0;
};
WsTable g_ws[kMaxDevices];

// A held slot: its buffer may be used until the holder is destroyed.
struct WsHold {
    std::shared_ptr<WsSlot> slot;
    std::unique_lock<std::mutex> held;
};

// The buffer of (current device, stream), at least `bytes` large, held for the caller.
int workspace(hipStream_t stream, size_t bytes, WsHold &hold, char **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxDevices) return MMBO_ERR_NO_DEVICE;
    WsTable &tab = g_ws[dev];
    for (;;) {
        std::shared_ptr<WsSlot> slot, victim;
        std::unique_lock<std::mutex> victim_held;
        {
            std::lock_guard<std::mutex> tl(tab.lock);
            for (auto &sl : tab.slots)
                if (sl->stream == stream) slot = sl;
            if (!slot) {
                if (tab.slots.size() >= kMaxWsSlots) {
                    // retire the least recently used slot that no call holds
                    size_t pick = tab.slots.size();
                    for (size_t i = 0; i < tab.slots.size(); ++i) {
                        if (pick < tab.slots.size() && tab.slots[i]->last_use >= tab.slots[pick]->last_use) continue;
                        std::unique_lock<std::mutex> t(tab.slots[i]->use, std::try_to_lock);
                        if (!t.owns_lock()) continue;
                        pick = i;
                        victim_held = std::move(t);
                    }
                    if (pick < tab.slots.size()) {
                        victim = tab.slots[pick];
                        victim->dead = true;
                        tab.slots.erase(tab.slots.begin() + (long)pick);
                    }
                    // (every slot held by a call in flight: the table grows past its bound for now)
                }
                slot = std::make_shared<WsSlot>();
                slot->stream = stream;
                tab.slots.push_back(slot);
            }
            slot->last_use = ++tab.clock;
        }
        if (victim) {
            if (victim->base) {
                e = hipDeviceSynchronize();
                (void)hipFree(victim->base);
                victim->base = nullptr;
                victim->bytes = 0;
            }
            victim_held.unlock();
            if (e != hipSuccess) return hip_fail(e);
        }
        std::unique_lock<std::mutex> held(slot->use);
        if (slot->dead) continue;                    // retired between the lookup and here: look the stream up again
        if (slot->bytes < bytes) {
            if (slot->base) {
                // earlier launches on this stream may still be using the old buffer (fails under stream capture: a captured
                // call must find its workspace already large enough, or use the entry point that allocates nothing)
                e = hipStreamSynchronize(stream);
                if (e != hipSuccess) return hip_fail(e);
                (void)hipFree(slot->base);
                slot->base = nullptr;
                slot->bytes = 0;
            }
            size_t want = std::max(bytes + bytes / 4, kWaveSumsBytes);
            void *p = nullptr;
            if (hipMalloc(&p, want) != hipSuccess) {
                (void)hipGetLastError();
                want = bytes;
                if (hipMalloc(&p, want) != hipSuccess) {
                    (void)hipGetLastError();
                    return MMBO_ERR_WORKSPACE;
                }
            }
            slot->base = static_cast<char *>(p);
            slot->bytes = want;
        }
        *out = slot->base;
        hold.slot = std::move(slot);
        hold.held = std::move(held);
        return MMBO_OK;
    }
}

// Takes the slots `which` selects out of the current device's table and frees their buffers.  `stream_only`: wait for
// that stream alone (its handle is still valid: the caller is about to destroy it); otherwise for the whole device.
int release_slots(bool stream_only, hipStream_t stream)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxDevices) return MMBO_ERR_NO_DEVICE;
    WsTable &tab = g_ws[dev];
    std::vector<std::shared_ptr<WsSlot>> out;
    {
        std::lock_guard<std::mutex> tl(tab.lock);
        for (size_t i = 0; i < tab.slots.size();) {
            if (!stream_only || tab.slots[i]->stream == stream) {
                out.push_back(tab.slots[i]);
                tab.slots.erase(tab.slots.begin() + (long)i);
            } else {
                ++i;
            }
        }
    }
    if (out.empty()) return MMBO_OK;
    hipError_t first = hipSuccess;
    for (auto &sl : out) {
        std::lock_guard<std::mutex> held(sl->use);       // a call that holds the slot queues its launches first
        sl->dead = true;
    }
    e = stream_only ? hipStreamSynchronize(stream) : hipDeviceSynchronize();
    if (e != hipSuccess) return hip_fail(e);
    for (auto &sl : out) {
        std::lock_guard<std::mutex> held(sl->use);
        if (sl->base) {
            e = hipFree(sl->base);
            if (e != hipSuccess && first == hipSuccess) first = e;
            sl->base = nullptr;
            sl->bytes = 0;
        }
    }
    return first == hipSuccess ? MMBO_OK : hip_fail(first);
}

// The workspace of the entry point that allocates nothing: one array per device in the library's own image, there from
// the moment the code object is loaded until the process ends.  In host code the array's name is only a handle: the
// device address of each GPU's copy comes from hipGetSymbolAddress, once per device, and that pointer is what the
// kernels get.  Nothing in it has to start at zero: every partial sum a GEMM reads was written by that same GEMM.
constexpr size_t kScratchPartialBytes = 32u << 20;
static __device__ __align__(256) unsigned char scratch[kScratchPartialBytes];
std::mutex g_scratch_mutex;
char *g_scratch_ptr[kMaxDevices] = {};

int static_scratch(char **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxDevices) return MMBO_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e);
        if (!p) return MMBO_ERR_WORKSPACE;
        g_scratch_ptr[dev] = static_cast<char *>(p);
    }
    *out = g_scratch_ptr[dev];
    return MMBO_OK;
}

// ---- table ------------------------------------------------------------------------------------
template <int DTYPE, int TILE>
hipError_t dispatch_tile(int tile, int ta, int tb, const GemmArgs &a, hipStream_t s)
{
    if (tile == TILE) return launch_staged<DTYPE, TILE>(ta, tb, a, s);
    if constexpr (TILE + 1 < NUM_TILES) return dispatch_tile<DTYPE, TILE + 1>(tile, ta, tb, a, s);
    return hipErrorInvalidValue;
}

template <int DTYPE, int TILE>
hipError_t dispatch_ring(int tile, int ta, int tb, const GemmArgs &a, hipStream_t s)
{
    if (tile == TILE) return launch_ring<DTYPE, TILE>(ta, tb, a, s);
    if constexpr (TILE + 1 < NUM_RING_TILES) return dispatch_ring<DTYPE, TILE + 1>(tile, ta, tb, a, s);
    return hipErrorInvalidValue;
}

template <int DTYPE, int TILE>
hipError_t dispatch_x16(int tile, int ta, int tb, const GemmArgs &a, hipStream_t s)
{
    if (tile == TILE) return launch_x16<DTYPE, TILE>(ta, tb, a, s);
    if constexpr (TILE + 1 < NUM_X16_TILES) return dispatch_x16<DTYPE, TILE + 1>(tile, ta, tb, a, s);
    return hipErrorInvalidValue;
}

template <int DTYPE, int TILE>
hipError_t dispatch_wave(int tile, int ta, int tb, const GemmArgs &a, int waves, hipStream_t s)
{
    if (tile == TILE) return launch_wave<DTYPE, TILE>(ta, tb, a, waves, s);
    if constexpr (TILE + 1 < wave_tiles(DTYPE)) return dispatch_wave<DTYPE, TILE + 1>(tile, ta, tb, a, waves, s);
    return hipErrorInvalidValue;
}

template <int TILE>
hipError_t dispatch_dots(int tile, int ta, int tb, const GemmArgs &a, hipStream_t s)
{
    if (tile == TILE) return launch_dots<TILE>(ta, tb, a, s);
    if constexpr (TILE + 1 < NUM_DOTS_TILES) return dispatch_dots<TILE + 1>(tile, ta, tb, a, s);
    return hipErrorInvalidValue;
}

template <int TILE>
hipError_t dispatch_planes(int tile, int ta, int tb, const GemmArgs &a, hipStream_t s)
{
    if (tile == TILE) return launch_planes<TILE>(ta, tb, a, s);
    if constexpr (TILE + 1 < NUM_PLANES_TILES) return dispatch_planes<TILE + 1>(tile, ta, tb, a, s);
    return hipErrorInvalidValue;
}

template <int TILE>
hipError_t dispatch_dgemm(int tile, int ta, int tb, const GemmArgs &a, hipStream_t s)
{
    if (tile == TILE) return launch_dgemm<TILE>(ta, tb, a, s);
    if constexpr (TILE + 1 < NUM_F64_TILES) return dispatch_dgemm<TILE + 1>(tile, ta, tb, a, s);
    return hipErrorInvalidValue;
}

template <int TILE>
int dgemm_lds_bytes_of(int tile)
{
    if (tile == TILE) return dgemm_lds_bytes<TILE>();
    if constexpr (TILE + 1 < NUM_F64_TILES) return dgemm_lds_bytes_of<TILE + 1>(tile);
    return 0;
}

template <int DTYPE, int TILE>
int lds_bytes_of(int tile)
{
    if (tile == TILE) return staged_lds_bytes<DTYPE, TILE>();
    if constexpr (TILE + 1 < NUM_TILES) return lds_bytes_of<DTYPE, TILE + 1>(tile);
    return 0;
}

inline size_t ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }

// Relative MFMA-pipe cost of a tile's inner loop (1.0 = the 256 x 256 tile): smaller wave tiles read more
// LDS per MFMA.  Fitted to sweeps of every config on MI355X.
double tile_cost(int dtype, int tile)
{
    static const double c32[NUM_TILES] = {1.00, 1.06, 1.03, 1.03, 1.08, 2.2};
    static const double c16[NUM_TILES] = {1.00, 1.10, 1.15, 1.25, 1.9, 4.0};
    return dtype == MMBO_F32 ? c32[tile] : c16[tile];
}

// Modelled time, in GPU clocks, of running the problem with the staged kernel of (tile, split).
// The staged kernel prefetches one stage ahead, so a stage costs the larger of its MFMA time (shared by the
// work-groups resident on the CU) and the global-load latency; short K and few tiles are latency-bound,
// which is what split-K and small tiles buy back.
double model_time(int dtype, int tile, int split, size_t m, size_t n, size_t k, int batch)
{
    const TileRow &r = tile_row(dtype, tile);
    const double cus = 256.0;
    const double mac_per_clk_cu = dtype == MMBO_F32 ? 128.0 : 2048.0;   // dense MFMA rate of one CU
    const double hbm_bytes_per_clk = 3300.0;                            // ~8 TB/s at ~2.4 GHz
    const double load_latency = 1700.0;                                 // clocks from issue to data in registers
    const double esz = dtype == MMBO_F32 ? 4.0 : 2.0;
    double tiles = (double)ceil_div(m, r.bm) * (double)ceil_div(n, r.bn) * batch * split;
    // work-groups resident per CU, bounded by LDS (160 KB) and by 2048 threads
    int lds = dtype == MMBO_F32 ? lds_bytes_of<0, 0>(tile) : lds_bytes_of<1, 0>(tile);
    int per_cu = 160 * 1024 / (lds > 0 ? lds : 1);
    int thr = r.wm * r.wn * 64;
    if (per_cu > 2048 / thr) per_cu = 2048 / thr;
    if (per_cu < 1) per_cu = 1;
    double slots = cus * per_cu;
    double rounds = (double)ceil_div((size_t)tiles, (size_t)slots);
    double resident = tiles >= slots ? per_cu : (tiles > cus ? tiles / cus : 1.0);   // tiles sharing one CU's pipes
    double stage_mfma = (double)r.bm * r.bn * r.bk * tile_cost(dtype, tile) / mac_per_clk_cu;
    double stage = stage_mfma * resident > load_latency ? stage_mfma * resident : load_latency;
    double stages = (double)ceil_div(ceil_div(k, (size_t)split), (size_t)r.bk);
    double epilogue = (double)r.bm * r.bn * esz * resident / 24.0;      // C tile through one CU's store path
    double compute = rounds * (stages * stage + load_latency + epilogue);
    double bytes = ((double)m * k + (double)k * n + (double)m * n) * batch * esz;
    double t = compute > bytes / hbm_bytes_per_clk ? compute : bytes / hbm_bytes_per_clk;
    t += 9000.0;                                                         // launch
    if (split > 1)   // second launch + partial sums written and read back
        t += 9000.0 + (double)m * n * batch * (2.0 * split * 4.0 + esz) / hbm_bytes_per_clk;
    return t;
}

// fp64: how many 64 x 64 tiles at the end of the walk go out as quarters: those behind the last whole round of the 256 CUs.
// 1152 x 2048 is 576 tiles, 2.25 to a CU: whole, they take as long as 3 rounds; the last 64 as 256 quarters, 2.25.  A quarter
// takes 0.3 of a tile's time (its operand traffic halves, its flops quarter), so up to three quarters to a CU, 192 tiles,
// are worth it, however many whole rounds precede them (aligned operands, us: 100 of 2 104.7 -> 88.4, 44 of 6 189.6 -> 167.5, 191 of
// 4 49.2 -> 48.0), but not three of them behind several rounds of a short k, where 0.9 of a tile's time is none to gain (145 of 5, TN 3648 x
// 1600 x 272 whole 62.0, quarters 64.1).  Fewer tiles than CUs are the 32 x 32 tile's.
constexpr int kQuarterTile = 3;
static_assert(kTilesF64[kQuarterTile].bm == 32 && kTilesF64[kQuarterTile].bn == 32, "a 64 x 64 tile's quarter");
size_t quartered_tiles(int tile, size_t tiles, int batch, size_t k)
{
    if (!dgemm_quarters(kTilesF64[tile].bm, kTilesF64[tile].bn) || batch != 1) return 0;
    const size_t rest = tiles % 256;
    if (rest > 128 && tiles >= 2 * 256 && tiles < 7 * 256 && k < 320) return 0;
    return tiles >= 256 && rest <= 192 ? rest : 0;
}

// fp64: does a grid of 64 x 64 tiles that ends in quarters stay with them, or do 32 x 32 tiles throughout take the call?  The model below
// compares rounds, but not how far the work-groups of a CU overlap: with few whole rounds all of them are resident at one time,
// start together and update C together, and 32 x 32 tiles, of which a CU runs some behind others, are as fast or faster on a short
// k or where the quarters fill a round badly.  Measured on 420 drawn shapes, quarters against 32 x 32 tiles, us (NT, C read): one round
// 5120 x 256 x 496 (one quarter to a CU) 26.6 / 26.9, but 27.2 / 26.6 with C not read, 1792 x 832 x 541 (two) 32.0 / 33.3, 2048 x 832 x 848 (three)
// 53.0 / 62.4, 896 x 1728 x 208 15.9 / 15.8; two rounds 1152 x 2048 x 384 (one) 34.7 / 34.8, 2112 x 1024 x 752 59.4 / 62.5, 960 x 2752 x 624 (three) 67.5 / 63.3;
// three 2432 x 1472 x 272 40.4 / 38.3, four 2304 x 2048 x 384 61.0 / 64.7, five 2432 x 2176 x 256 49.3 / 51.7.  The pick is then within 0.6 % of the
// faster of the two on average, 4 % at worst on aligned operands.
bool quarters_pay(size_t tiles, size_t k)
{
    const size_t whole = tiles / 256, quarters = ceil_div(tiles % 256, 64);
    if (whole == 1) return quarters >= 2 && k >= 256;
    if (whole == 2) return quarters < 3 && k >= 256;
    return whole >= 5 || k >= 320;
}

// fp64: microseconds.  Work-groups run in rounds of (CUs x work-groups per CU); a tile costs a fixed overhead
// (first stage, C update, dispatch of its successor: measured per tile and CU with K swept from 96 to 1536 on the
// HPL shape's M and N) plus its K at the tile's in-loop efficiency (from 8192^3), both shared by the work-groups
// resident on the CU; the last, partial round runs with fewer of them, or as quarters that cost what the 32 x 32 tile does
// (drawn shapes that end so: within 12 % of the measured time, 16 % where C is read).
double model_time_f64(int tile, size_t m, size_t n, size_t k, int batch)
{
    //                                    128x128/4w 256x128/8w 64x64  32x32  128x128/8w 128x64
    static const double overhead_us[NUM_F64_TILES] = {12.8, 26.5, 1.54, 0.25, 10.6, 5.9};
    static const double in_loop_eff[NUM_F64_TILES] = {0.89, 0.853, 0.846, 0.704, 0.91, 0.84};
    static const int resident[NUM_F64_TILES] = {2, 1, 5, 8, 2, 3};
    const TileRow &r = kTilesF64[tile];
    const double cus = 256.0, flop_per_us_cu = 78.6e6 / 256.0, launch = 5.0;
    const double tiles = (double)ceil_div(m, r.bm) * (double)ceil_div(n, r.bn) * batch;
    auto tile_us = [&](int t) {
        return overhead_us[t] + 2.0 * kTilesF64[t].bm * kTilesF64[t].bn * (double)(k ? k : 1) / flop_per_us_cu / in_loop_eff[t];
    };
    const double per_tile = tile_us(tile);
    if (const size_t rest = quartered_tiles(tile, (size_t)tiles, batch, k))
        return launch + std::floor(tiles / cus) * per_tile + std::ceil(4.0 * (double)rest / cus) * tile_us(kQuarterTile);
    const double slots = cus * resident[tile];
    const double full = std::floor(tiles / slots), last = tiles - full * slots;
    double t = launch + full * per_tile * resident[tile];
    if (last > 0) t += per_tile * std::ceil(last / cus);
    return t;
}

}  // namespace

hipError_t launch_splitk_reduce(int dtype, const GemmArgs &args, hipStream_t stream)
{
    size_t mn = (size_t)args.m * args.n;
    const bool vec = args.m % 4 == 0;      // a thread then owns 16 bytes of sums of one column
    const size_t groups = vec ? mn / 4 : mn;
    // more than sixteen splits: several threads share the splits of one group (see the kernel)
    GemmArgs a = args;
    a.reduce_parts = args.splits <= 16 ? 1 : args.splits <= 32 ? 4 : 8;
    dim3 grid((unsigned)ceil_div(groups * a.reduce_parts, 256), 1, args.batch);
    auto launch = [&](auto zero) {
        using T = decltype(zero);
        if (a.reduce_parts == 1)
            return vec ? launch_kernel(splitk_reduce_kernel<T, true, false>, grid, dim3(256), 0, stream, a)
                       : launch_kernel(splitk_reduce_kernel<T, false, false>, grid, dim3(256), 0, stream, a);
        return vec ? launch_kernel(splitk_reduce_kernel<T, true, true>, grid, dim3(256), 0, stream, a)
                   : launch_kernel(splitk_reduce_kernel<T, false, true>, grid, dim3(256), 0, stream, a);
    };
    return dtype == MMBO_F32 ? launch(0.0f) : launch((half_t)0.0f);           // (fp64 calls never split k over work-groups)
}

}  // namespace mmbo

using namespace mmbo;

extern "C" {

const char *mmbo_version(void) { return "mmbo_gemm 0.1 (gfx950)"; }

int mmbo_last_hip_error(void) { return g_last_hip_error; }

const char *mmbo_status_string(int status)
{
    switch (status) {
        case MMBO_OK: return "ok";
        case MMBO_ERR_INVALID_DTYPE: return "invalid dtype";
        case MMBO_ERR_INVALID_OP: return "invalid transpose op";
        case MMBO_ERR_INVALID_SIZE: return "invalid size, leading dimension, stride or batch";
        case MMBO_ERR_NULL_POINTER: return "null pointer";
        case MMBO_ERR_INVALID_CONFIG: return "invalid config id";
        case MMBO_ERR_HIP: return "HIP runtime error";
        case MMBO_ERR_NO_DEVICE: return "no usable device";
        case MMBO_ERR_WORKSPACE: return "split-K workspace allocation failed";
        default: return "unknown status";
    }
}

int mmbo_num_configs(int dtype)
{
    if (!valid_dtype(dtype)) return -MMBO_ERR_INVALID_DTYPE;
    return dtype == MMBO_F64 ? NUM_F64_TILES : num_configs(dtype);
}

static void describe_planes(int tile, int split, mmbo_config_desc *out)
{
    const PlanesRow &r = kPlanesTiles[tile];
    std::memset(out, 0, sizeof(*out));
    std::snprintf(out->name, sizeof(out->name), "MT%03dx%03dx%02d_WT%03dx%03d_W%d_GSU%02d_LSU%02d_BF16X3", r.bm, r.bn, kPlanesBk, r.bm / r.wm,
                  r.bn / r.wn, r.wm * r.wn * r.kg, split, r.kg);
    out->macro_tile_m = r.bm;
    out->macro_tile_n = r.bn;
    out->depth_u = kPlanesBk;
    out->threads = r.wm * r.wn * r.kg * 64;
    out->wave_tile_m = r.bm / r.wm;
    out->wave_tile_n = r.bn / r.wn;
    out->split_k = split;
    out->lds_bytes = r.kg * 2 * 3 * (r.bm + r.bn) * 64;
}

int mmbo_config_info(int dtype, int config_id, mmbo_config_desc *out)
{
    if (!valid_dtype(dtype)) return MMBO_ERR_INVALID_DTYPE;
    if (!out) return MMBO_ERR_NULL_POINTER;
    if (config_id < 0 || config_id >= mmbo_num_configs(dtype)) return MMBO_ERR_INVALID_CONFIG;
    std::memset(out, 0, sizeof(*out));
    if (dtype == MMBO_F64) {
        const TileRow &r = kTilesF64[config_id];
        std::snprintf(out->name, sizeof(out->name), "MT%03dx%03dx%02d_WT%03dx%03d_W%d_GSU01_MFMA16x16x4", r.bm, r.bn,
                      r.bk, r.bm / r.wm, r.bn / r.wn, r.wm * r.wn);
        out->macro_tile_m = r.bm; out->macro_tile_n = r.bn; out->depth_u = r.bk; out->threads = r.wm * r.wn * 64;
        out->wave_tile_m = r.bm / r.wm; out->wave_tile_n = r.bn / r.wn; out->split_k = 1;
        out->lds_bytes = dgemm_lds_bytes_of<0>(config_id);
        return MMBO_OK;
    }
    const ConfigRef c = config_ref(config_id);
    if (c.planes) {
        describe_planes(c.tile, c.split, out);
        return MMBO_OK;
    }
    if (c.ring) {
        const RingRow &r = c.x16 ? kX16Tiles[c.tile] : kRingTiles[c.tile];
        std::snprintf(out->name, sizeof(out->name), "MT%03dx%03dx%02d_WT%03dx%03d_W%d_GSU%02d_DTL1_RING%d%s", r.bm, r.bn,
                      ring_bk(dtype), r.bm / r.wm, r.bn / r.wn, r.wm * r.wn, c.split, r.depth,
                      !c.x16 ? "" : dtype == MMBO_F16 ? "_MFMA16x16x32_ACC" : "_MFMA16x16x4_ACC");
        out->macro_tile_m = r.bm;
        out->macro_tile_n = r.bn;
        out->depth_u = ring_bk(dtype);
        out->threads = r.wm * r.wn * 64;
        out->wave_tile_m = r.bm / r.wm;
        out->wave_tile_n = r.bn / r.wn;
        out->split_k = c.split;
        out->lds_bytes = r.depth * (r.bm + r.bn) * 64;
        return MMBO_OK;
    }
    int tile = config_id % NUM_TILES, split = kSplits[config_id / NUM_TILES];
    const TileRow &r = tile_row(dtype, tile);
    std::snprintf(out->name, sizeof(out->name), "MT%03dx%03dx%02d_WT%03dx%03d_W%d_GSU%02d", r.bm, r.bn, r.bk,
                  r.bm / r.wm, r.bn / r.wn, r.wm * r.wn, split);
    out->macro_tile_m = r.bm;
    out->macro_tile_n = r.bn;
    out->depth_u = r.bk;
    out->threads = r.wm * r.wn * 64;
    out->wave_tile_m = r.bm / r.wm;
    out->wave_tile_n = r.bn / r.wn;
    out->split_k = split;
    out->lds_bytes = dtype == MMBO_F32 ? lds_bytes_of<0, 0>(tile) : lds_bytes_of<1, 0>(tile);
    return MMBO_OK;
}

static TileRow planes_tile(int tile) { return TileRow{kPlanesTiles[tile].bm, kPlanesTiles[tile].bn, kPlanesBk, 0, 0}; }

// Macro tile (and depthU) of a config id.
static TileRow config_tile(int dtype, int id)
{
    if (dtype == MMBO_F64) return kTilesF64[id];
    const ConfigRef c = config_ref(id);
    if (c.planes) return planes_tile(c.tile);
    if (!c.ring) return tile_row(dtype, c.tile);
    const RingRow &rr = c.x16 ? kX16Tiles[c.tile] : kRingTiles[c.tile];
    return TileRow{rr.bm, rr.bn, ring_bk(dtype), 0, 0};
}

// Per-thread global offsets are 32-bit: one tile's span of an operand must stay below 2 GiB.
static bool tile_span_ok(const TileRow &r, int transA, int transB, size_t lda, size_t ldb, size_t esz)
{
    size_t span_a = (transA ? (size_t)r.bm : (size_t)r.bk) * lda * esz;
    size_t span_b = (transB ? (size_t)r.bk : (size_t)r.bn) * ldb * esz;
    return span_a < 0x7FFFFF00ull && span_b < 0x7FFFFF00ull;
}

// Modelled time, in microseconds, of a whole-tile kernel (ring or x16 family, ring tile index rt: 256x256, 128x128,
// 128x64, 64x64) on a shape made of whole tiles.  Work-groups run in rounds of (CUs x work-groups per CU); a tile costs
// a ring fill, its slices at the family's in-loop efficiency (shared by the work-groups resident on the CU) and its
// C traffic; the last, partial round runs with fewer work-groups per CU; split-K adds the reduction launch.  The
// constants are a least-squares fit to the times of every such config on 45 shapes (gemm_mmbo_amd/tune.py --dump);
// on those shapes the model's pick is within 2.5 % of the fastest config on average, 21 % at worst.
// split_lines: the rows of a packed operand (leading dimension = its stored row count) do not start on 128-byte lines,
// so every request of the direct loads touches one line more.  Measured on fp16: the 128 x 128 and smaller tiles, which
// are bound by that stream, lose 13-26 % of their in-loop rate (3000^3 against 3072^3, 4104^3 against 4096^3, 8200 against
// 8192), the 256 x 256 tile up to 15 % at 3000 and nothing at 4104 or 8200; fp32 tiles, MFMA-bound, lose nothing.
static double model_time_tile(int dtype, const RingRow &r, double e, int split, size_t m, size_t n, size_t k, int batch)
{
    const double launch = 5.9, fill = 0.65, c_us_per_kb = 0.0272, reduce_launch = 1.43, reduce_us_per_mb = 0.28;
    const double esz = dtype == MMBO_F32 ? 4.0 : 2.0;
    const double flop_per_us_cu = dtype == MMBO_F32 ? 0.614e6 : 9.83e6;             // matrix peak of one CU
    const int bk = ring_bk(dtype);
    const int lds = r.depth * (r.bm + r.bn) * 64;
    int per_cu = 160 * 1024 / lds;
    if (per_cu > 3) per_cu = 3;
    if (per_cu < 1) per_cu = 1;
    const double cus = 256.0;
    const double wgs = (double)ceil_div(m, (size_t)r.bm) * (double)ceil_div(n, (size_t)r.bn) * split * batch;
    const double slices = std::ceil(std::ceil((double)k / bk) / split);
    auto tile_time = [&](double resident) {
        return fill + slices * (2.0 * r.bm * r.bn * bk / flop_per_us_cu) * resident / e +
               c_us_per_kb * r.bm * r.bn * esz * resident / 1e3;
    };
    const double slots = cus * per_cu;
    const double full = std::floor(wgs / slots), last = wgs - full * slots;
    double t = launch + full * tile_time(per_cu);
    if (last > 0) {
        // A last round that leaves CUs idle runs faster per tile on fp16: the chip is power-limited on these MFMAs and the
        // clock rises when fewer CUs draw power (HGEMM 3072^3 on 144 tiles of 256 x 256: 54 us against 74 us for a full
        // round of the same tiles; 5120^3, 256 + 144 tiles: the second round takes 0.82 of the first).
        // (with several work-groups to a CU the round lasts as long as the fullest CU's; "busy" is the share of CU time in use)
        const double busy = last / (cus * std::ceil(last / cus));
        // (the tiles that run one to a CU are the power-limited ones; the smaller ones, bound by the L2 -> LDS stream, gain
        // less: HGEMM 1280 x 1280 x 4096 on 100 tiles of 128 x 128 runs at 0.86 of a full round's time per tile)
        const bool one_per_cu = r.depth * (r.bm + r.bn) * 64 > 80 * 1024;
        const double boost = dtype != MMBO_F16 ? 1.0 : one_per_cu ? 0.45 + 0.55 * busy : 0.7 + 0.3 * busy;
        t += tile_time(std::ceil(last / cus)) * boost;
    }
    if (split > 1) t += reduce_launch + reduce_us_per_mb * (double)m * n * batch * (split * 4.0 + esz) / 1e6;
    return t;
}
static double model_time_ring(int dtype, bool x16, int rt, int split, size_t m, size_t n, size_t k, int batch,
                              bool split_lines = false)
{
    static const double eff[2][2][NUM_RING_TILES] = {
        // 256x256 128x128 128x64  64x64
        {{0.9451, 0.9134, 0.8667, 0.9015}, {0.9387, 0.9039, 0.8402, 0.8561}},       // fp32: ring, x16
        {{0.5607, 0.3426, 0.2795, 0.2658}, {0.5879, 0.4873, 0.3151, 0.2560}},       // fp16: ring, x16
    };
    double e = eff[dtype == MMBO_F32 ? 0 : 1][x16 ? 1 : 0][rt];
    if (split_lines && dtype == MMBO_F16) e *= rt == 0 ? 0.95 : 0.78;
    return model_time_tile(dtype, kRingTiles[rt], e, split, m, n, k, batch);      // the x16 tiles of the same macro tile have the same depth
}
// The x16 kernel's tiles without a ring-kernel twin: 192 x 192, 256 x 192, 192 x 256 (kX16Tiles[5..7]).  In-loop
// efficiency: 192 x 192 from HGEMM 6144^3 (four whole rounds, 381 us) and SGEMM 3072^3 (one round, 404 us); the two
// rectangular ones between that and the 256 x 256 tile's.
constexpr int kFirstX16OnlyTile = 5;
static double model_time_x16_only(int dtype, int tile, int split, size_t m, size_t n, size_t k, int batch, bool split_lines)
{
    static const double eff16[3] = {0.50, 0.55, 0.55}, eff32[3] = {0.93, 0.935, 0.935};
    double e = (dtype == MMBO_F32 ? eff32 : eff16)[tile - kFirstX16OnlyTile];
    if (split_lines && dtype == MMBO_F16) e *= 0.90;
    return model_time_tile(dtype, kX16Tiles[tile], e, split, m, n, k, batch);
}

// The cost model's pick among the staged configs (fp32/fp16), which take any shape and any alignment.
static int select_staged(int dtype, size_t m, size_t n, size_t k, int batch, double *us = nullptr)
{
    int best = 0;
    double best_t = 0.0;
    for (int si = 0; si < NUM_SPLITS; ++si) {
        int split = kSplits[si];
        for (int tile = 0; tile < NUM_TILES; ++tile) {
            const TileRow &r = tile_row(dtype, tile);
            if (split > 1 && ceil_div(k, (size_t)split) < (size_t)2 * r.bk) continue;   // slices too thin
            double t = model_time(dtype, tile, split, m, n, k ? k : 1, batch);
            if (best_t == 0.0 || t < best_t) { best_t = t; best = tile + NUM_TILES * si; }
        }
    }
    if (us) *us = best_t / 2400.0;
    return best;
}

// The pick of mmbo_select_config and, in *us, the microseconds its model (or the tuned table's record) gives it.
static int select_config(int dtype, int transA, int transB, size_t m, size_t n, size_t k, int batch, double *us)
{
    *us = 0.0;
    if (!valid_dtype(dtype)) return -MMBO_ERR_INVALID_DTYPE;
    if ((transA | transB) & ~1) return -MMBO_ERR_INVALID_OP;
    if (batch < 0) return -MMBO_ERR_INVALID_SIZE;
    if (m == 0 || n == 0 || batch == 0) return 0;
    for (const TunedRow &t : kTuned)
        if (t.dtype == dtype && t.transA == transA && t.transB == transB && t.m == m && t.n == n && t.k == k &&
            t.batch == batch) {
            *us = 2.0 * (double)m * (double)n * (double)k * batch / t.tflops * 1e-6;
            return t.config_id;
        }
    if (dtype == MMBO_F64) {
        int best = 0;
        double best_t = 0.0;
        for (int tile = 0; tile < NUM_F64_TILES; ++tile) {
            double t = model_time_f64(tile, m, n, k, batch);
            if (best_t == 0.0 || t < best_t) { best_t = t; best = tile; }
        }
        const size_t tiles = ceil_div(m, kTilesF64[best].bm) * ceil_div(n, kTilesF64[best].bn);
        if (quartered_tiles(best, tiles, batch, k) > 0 && !quarters_pay(tiles, k)) {
            best = kQuarterTile;
            best_t = model_time_f64(best, m, n, k, batch);
        }
        *us = best_t;
        return best;
    }
    // Whole-tile kernels (deeper prefetch, no edge handling) measured faster than the staged kernel on every shape
    // they apply to: where one applies, the fastest of them by model_time_ring takes the call.  fp16: the x16 family
    // (16x16x32 MFMAs), except that the 64 x 64 tile is faster on 32x32x16; fp32: the ring family, except that the
    // x16 kernel's 256 x 256 tile (v_mfma_f32_16x16x4_f32, four wavefronts) measures 1.5-2 % faster than the ring
    // kernel's at 8192^3 in NN, TN and TT (0.8 % slower in NT).
    {
        static const int x16_of_ring[NUM_RING_TILES] = {0, 2, 3, 4};       // same macro tile in kX16Tiles (256 x 256: four wavefronts)
        int pick = -1;
        double pick_t = 0.0;
        const size_t esz = dtype == MMBO_F32 ? 4 : 2;
        const bool split_lines = ((transA ? k : m) * esz) % 128 != 0 || ((transB ? n : k) * esz) % 128 != 0;
        for (int rt = 0; rt < NUM_RING_TILES; ++rt)
            for (int si = 0; si < NUM_SPLITS; ++si) {
                const bool ring_ok = ring_shape_ok(dtype, rt, kSplits[si], transA, transB, m, n, k, false);
                const bool x16_ok = ring_shape_ok(dtype, x16_of_ring[rt], kSplits[si], transA, transB, m, n, k, true);
                if (!ring_ok && !x16_ok) continue;
                // A dimension smaller than the tile: only the 64 x 64 fp16 tile on a long k is worth it (measured against
                // the staged kernel's 32 x 32 tile: HGEMM 16 x 4096 x 4096 11.8 against 17.5 us, 48 x 48 x 8192 10.1
                // against 17.1, 32 x 8192 x 1024 9.1 against 8.5-9.4; SGEMM 4096 x 32 x 4096 27.4 against 22.9).
                if (!ring_ok && (m < (size_t)kRingTiles[rt].bm || n < (size_t)kRingTiles[rt].bn) &&
                    !(dtype == MMBO_F16 && rt == 3 && k >= 1024))
                    continue;
                if (kSplits[si] > 1 && (k / ring_bk(dtype)) / (size_t)kSplits[si] < 2) continue;      // slices too thin
                if ((size_t)batch * kSplits[si] > 65535) continue;
                bool x16 = dtype == MMBO_F16 ? rt != 3 : (rt == 0 && !(transA == 0 && transB == 1));
                if (!ring_ok) x16 = true;           // ragged M or N: only the x16 kernel has edge tiles
                if (!x16_ok) x16 = false;
                const double t = model_time_ring(dtype, x16, rt, kSplits[si], m, n, k, batch, split_lines);
                if (pick < 0 || t < pick_t) {
                    pick_t = t;
                    pick = x16 ? x16_config_id(x16_of_ring[rt], si) : ring_config_id(rt, si);
                }
            }
        // the 192-row and 192-column tiles: where they fill the rounds of 256 CUs better than the power-of-two tiles do
        static_assert(kX16Tiles[kFirstX16OnlyTile].bm == 192 && kX16Tiles[kFirstX16OnlyTile].bn == 192 && NUM_X16_TILES == 8,
                      "x16 tiles 5, 6, 7 are 192 x 192, 256 x 192, 192 x 256");
        for (int tile = kFirstX16OnlyTile; tile < NUM_X16_TILES; ++tile) {
            if (m < (size_t)kX16Tiles[tile].bm || n < (size_t)kX16Tiles[tile].bn) continue;
            for (int si = 0; si < NUM_SPLITS; ++si) {
                if (!ring_shape_ok(dtype, tile, kSplits[si], transA, transB, m, n, k, true)) continue;
                if (kSplits[si] > 1 && (k / ring_bk(dtype)) / (size_t)kSplits[si] < 2) continue;
                if ((size_t)batch * kSplits[si] > 65535) continue;
                const double t = model_time_x16_only(dtype, tile, kSplits[si], m, n, k, batch, split_lines);
                if (pick < 0 || t < pick_t) {
                    pick_t = t;
                    pick = x16_config_id(tile, si);
                }
            }
        }
        if (pick >= 0) {
            *us = pick_t;
            return pick;
        }
    }
    return select_staged(dtype, m, n, k, batch, us);
}

int mmbo_select_config(int dtype, int transA, int transB, size_t m, size_t n, size_t k, int batch)
{
    double us;
    return select_config(dtype, transA, transB, m, n, k, batch, &us);
}

int mmbo_wg_remap(unsigned linear_id, unsigned nwg0, unsigned nwg1, unsigned wgm, unsigned num_xcd,
                  unsigned *wg0, unsigned *wg1)
{
    if (!wg0 || !wg1) return MMBO_ERR_NULL_POINTER;
    if (nwg0 == 0 || nwg1 == 0 || wgm == 0 || num_xcd == 0) return MMBO_ERR_INVALID_SIZE;
    if ((unsigned long long)nwg0 * nwg1 > 0xFFFFFFFFull || linear_id >= nwg0 * nwg1) return MMBO_ERR_INVALID_SIZE;
    uint32_t a, b;
    wg_remap(linear_id, nwg0, nwg1, wgm, num_xcd, a, b);
    *wg0 = a;
    *wg1 = b;
    return MMBO_OK;
}

int mmbo_chip_block_remap(unsigned linear_id, unsigned nwg0, unsigned nwg1, unsigned *wg0, unsigned *wg1)
{
    if (!wg0 || !wg1) return MMBO_ERR_NULL_POINTER;
    if (nwg0 < 16 || nwg1 < 16) return MMBO_ERR_INVALID_SIZE;
    if ((unsigned long long)nwg0 * nwg1 > 0xFFFFFFFFull || linear_id >= nwg0 * nwg1) return MMBO_ERR_INVALID_SIZE;
    uint32_t a, b;
    chip_block_remap(linear_id, nwg0, nwg1, a, b);
    *wg0 = a;
    *wg1 = b;
    return MMBO_OK;
}

int mmbo_batch_xcd_remap(unsigned linear_id, unsigned tiles, unsigned batch, unsigned *tile, unsigned *batch_index)
{
    if (!tile || !batch_index) return MMBO_ERR_NULL_POINTER;
    if (tiles == 0 || batch == 0 || batch % 8 != 0) return MMBO_ERR_INVALID_SIZE;
    if ((unsigned long long)tiles * batch > 0xFFFFFFFFull || linear_id >= tiles * batch) return MMBO_ERR_INVALID_SIZE;
    uint32_t t, z;
    batch_xcd_remap(linear_id, tiles, 8, t, z);
    *tile = t;
    *batch_index = z;
    return MMBO_OK;
}

int mmbo_release_workspace(void) { return release_slots(false, nullptr); }

int mmbo_release_stream_workspace(void *stream) { return release_slots(true, static_cast<hipStream_t>(stream)); }

int mmbo_workspace_info(size_t *slots, size_t *bytes)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxDevices) return MMBO_ERR_NO_DEVICE;
    WsTable &tab = g_ws[dev];
    std::lock_guard<std::mutex> tl(tab.lock);
    size_t total = 0;
    for (auto &sl : tab.slots) total += sl->bytes;          // (a size being changed right now may be read stale: a diagnostic)
    if (slots) *slots = tab.slots.size();
    if (bytes) *bytes = total;
    return MMBO_OK;
}

size_t mmbo_static_workspace_bytes(void) { return kScratchPartialBytes; }

}  // extern "C"

namespace {

// Where the partial sums of a split-K config go.
enum class WsSource { kLibrary, kStatic };

// ---- the automatic pick between a config of the tables and the split-by-wavefront kernel ------------------------------

struct WavePick {
    int tile;           // row of kWaveTiles; < 0: none
    int waves, split;
    double us;          // modelled
};

// Modelled microseconds of the split-by-wavefront kernel.  A work-group costs a start, its slices -- each as long as the
// slower of its wavefronts' MFMAs and LDS reads, of the memory lines the CU's wavefronts pull through its vector path, and of
// the lines all CUs pull -- and its part of C; work-groups run in rounds of as many as LDS lets share a CU; the whole takes
// at least what its bytes take from memory, and a call what the host takes to launch it.  Constants: least squares over 540
// drawn shapes x every (tile, wavefronts, splits) that fits them; the pick is within 4 - 5 % of the fastest of them on
// average, 39 % at worst.
struct WaveModel {
    double launch, start;           // us
    double mfma_eff, clk_per_read;  // MFMA rate reached in the loop; clocks per LDS fragment read
    double gap;                     // us per slice of a wavefront that has its SIMD to itself
    double round_trip;              // us from a slice's request to its use, shared by the pairs in flight
    double cu_bytes, chip_bytes;    // bytes of lines per us: one CU's path, all CUs together
    double hbm_bytes;               // bytes per us from memory
    double c_cu, c_wave;            // us per 1024 elements of a tile's C: through the CU, through each wavefront
    double tail;                    // us for a partial slice through registers
    double reduce, reduce_per_mb;   // us: second launch; per MB of partial sums
};
constexpr WaveModel kWaveModel[3] = {
    {2.25, 1.08, 0.899, 7.4, 0.023, 0.372, 108.4e3, 31.9e6, 5.25e6, 0.322, 0.516, 0.376, 2.08, 0.370},      // fp32
    {2.51, 0.65, 0.421, 0.0, 0.036, 0.233, 122.7e3, 32.8e6, 5.69e6, 0.193, 1.173, 0.731, 1.68, 0.379},      // fp16
    {2.03, 1.15, 0.734, 8.9, 0.026, 0.471, 98.6e3, 26.0e6, 5.58e6, 0.484, 0.444, 0.246, 0.0, 0.0},        // fp64 (never a second launch)
};

struct WaveShape {
    int dtype, transA, transB;
    size_t m, n, k;
    int batch;
    size_t lda, ldb;
    bool read_c;
    bool wide_c;        // C is read, and its columns (256 rows or more) lie at least four times their own length apart
};
WaveShape wave_shape(int dtype, int transA, int transB, size_t m, size_t n, size_t k, int batch, size_t lda, size_t ldb, size_t ldc, bool read_c)
{
    return {dtype, transA, transB, m, n, k, batch, lda, ldb, read_c, read_c && m >= 256 && ldc >= 4 * m};
}

// us that one slice takes a SIMD: its MFMAs and LDS reads
double wave_slice_work_us(const WaveShape &p, int tile)
{
    const WaveModel &w = kWaveModel[p.dtype];
    const WaveRow &row = kWaveTiles[tile];
    const int reads_rc = p.dtype == MMBO_F32 ? 4 : 2;
    const double reads = row.bm / 16 * (p.transA ? 1 : reads_rc) + row.bn / 16 * (p.transB ? reads_rc : 1);
    const double clocks = (p.dtype == MMBO_F16 ? 16.0 : 128.0) * (row.bm / 16) * (row.bn / 16);
    return (clocks / w.mfma_eff + reads * w.clk_per_read) / 2400.0;
}

double wave_model_us(const WaveShape &p, int tile, int waves, int split)
{
    const WaveModel &w = kWaveModel[p.dtype];
    const WaveRow &row = kWaveTiles[tile];
    const double esz = p.dtype == MMBO_F64 ? 8 : p.dtype == MMBO_F32 ? 4 : 2, sum_size = p.dtype == MMBO_F64 ? 8 : 4;
    const size_t bk = (size_t)(64 / esz);
    const size_t pairs = ceil_div(ceil_div(p.k, bk), 2), pairs_per_split = ceil_div(pairs, (size_t)split), splits = ceil_div(pairs, pairs_per_split);
    const double slices = (double)std::min(2 * ceil_div(pairs_per_split, (size_t)waves), ceil_div(p.k, bk));
    const double wgs = (double)(ceil_div(p.m, row.bm) * ceil_div(p.n, row.bn) * splits) * p.batch;
    const double ring = row.depth * (row.bm + row.bn) * 64.0, partial = (row.bm + 16 / sum_size) * row.bn * sum_size;
    const int per_cu = std::max(1, std::min((int)(160 * 1024 / (waves * std::max(ring, partial))), 16 / waves));
    // bytes of 128-byte lines one slice of an operand touches: whole lines where rows start on them, more where they do not
    auto lines = [&](size_t rows, size_t dim, bool k_contiguous, size_t ld) {
        const double here = (double)std::min(rows, ceil_div(dim, (size_t)16) * 16);
        const bool on_lines = (size_t)(ld * esz) % 128 == 0;
        if (k_contiguous) return here * 64 * (on_lines ? 1.0 : 1.5);
        const double width = here * esz, per_column = on_lines ? std::max(width, 128.0) : width + 112;
        return per_column * 64 / esz;
    };
    const double line_bytes = lines(row.bm, p.m, p.transA, p.lda) + lines(row.bn, p.n, !p.transB, p.ldb);
    const double work = wave_slice_work_us(p, tile);
    const size_t per16 = (size_t)(16 / esz);
    const bool tail = p.k % bk != 0 || (!p.transA && p.m % per16 != 0) || (p.transB && p.n % per16 != 0);
    auto round = [&](double on_cu, double on_chip) {
        const double slice = std::max(std::max(work * std::ceil(on_cu * waves / 4.0), std::max(work + w.gap, w.round_trip * 2 / row.depth)),
                                      std::max(line_bytes * on_cu * waves / w.cu_bytes, line_bytes * waves * on_chip / w.chip_bytes));
        return w.start + slices * slice + row.bm * row.bn * (w.c_cu * on_cu + w.c_wave / waves) / 1024 + (tail ? w.tail : 0.0);
    };
    const double slots = 256.0 * per_cu, full = std::floor(wgs / slots), last = wgs - full * slots;
    double t = full * round(per_cu, slots);
    if (last > 0) t += round(std::ceil(last / 256), last);
    const double bytes = p.batch * ((double)p.m * p.k + (double)p.k * p.n + (double)p.m * p.n * (p.read_c ? 2 : 1)) * esz;
    const double memory = bytes / w.hbm_bytes + 0.5 * w.start;
    t = std::max(t, memory) + 0.15 * std::min(t, memory) + w.launch;
    double host = 5.1;
    if (splits > 1) {
        t += w.reduce + w.reduce_per_mb * p.batch * (double)p.m * p.n * sum_size * splits / 1e6;
        host = 8.8;
    }
    return std::max(t, host) + 0.02 * std::min(t, host);
}

// may_split: k may also be split over work-groups (GlobalSplitU: a workspace and a second launch).  Only where the pick of
// mmbo_select_config splits as well: a caller reads from that pick whether a call uses a workspace -- whether two calls of the
// entry point that allocates nothing may overlap, whether a call needs memory of its own before it can be captured.
// Only a pick below `limit` microseconds.
WavePick pick_wave(const WaveShape &p, bool may_split, double limit = 1e300)
{
    WavePick best{-1, 0, 0, limit};
    const double esz = p.dtype == MMBO_F64 ? 8 : p.dtype == MMBO_F32 ? 4 : 2;
    const size_t slices = ceil_div(p.k, (size_t)(64 / esz));
    if (p.k == 0) return best;
    for (int tile = 0; tile < wave_tiles(p.dtype); ++tile) {
        const size_t tiles = ceil_div(p.m, kWaveTiles[tile].bm) * ceil_div(p.n, kWaveTiles[tile].bn);
        if (tiles > 65535) continue;
        // (the slices' work alone, spread over all SIMDs, however k is split: most tiles, and most large calls, need no more than this)
        if ((kWaveModel[p.dtype].launch + (double)slices * tiles * p.batch * wave_slice_work_us(p, tile) / 1024.0) * 0.999999 >= best.us) continue;
        for (int waves : {1, 4, 8}) {
            if (waves > 1 && slices < (size_t)waves) continue;
            if (waves > wave_max_waves(kWaveTiles[tile])) continue;
            for (int split = 1; split <= (may_split ? 64 : 1); split *= 2) {
                // (splits: at least a pair of slices per wavefront, not beyond what the chip holds at one time; the partial sums
                // then fit the static workspace, so that both entry points run the same split)
                if (split > 1 && (slices < (size_t)split * waves * 2 || tiles * p.batch * split > kMaxSplitWaveGroups))
                    break;
                const double us = wave_model_us(p, tile, waves, split);
                if (us < best.us) best = WavePick{tile, waves, split, us};
            }
        }
    }
    return best;
}

// What the pick of mmbo_select_config takes, in place of the `us` of that pick's model.  The staged kernel's: the model knows the tiles of a few
// large problems; the calls that still come to this kernel are batches of narrow problems and operands with less than 16 bytes of m or
// n in memory, whose rounds of short work-groups, and whose loads by elements where columns start off 16 bytes, take up to seven times as
// long as it says.  Least squares over the times of 828 such drawn calls (fp16 574, fp32 254): 17 - 21 % rms, 24 - 45 % without.
bool is_staged(int dtype, int config_id)
{
    if (dtype == MMBO_F64) return false;
    const ConfigRef c = config_ref(config_id);
    return !c.ring && !c.planes;
}
// fp64's, for its 32 x 32 and 64 x 64 tiles: the model shares the MFMAs' time out, but a slice of 16 k takes a work-group a round trip however idle
// its CU is.  us per slice, 2,600 drawn calls: 32 x 32 with up to three work-groups per CU 0.35 - 0.39 (128 slices and more, whose operands the L2
// does not hold, 0.57 - 0.60), where the model says 0.16 for one; 64 x 64 with one 0.70 - 0.75 (0.78).
double config_us(const WaveShape &p, int config_id, double us)
{
    if (p.dtype == MMBO_F64) {
        const int bm = kTilesF64[config_id].bm, bn = kTilesF64[config_id].bn;
        const size_t slices = ceil_div(p.k, (size_t)16);
        if (bm != bn || bm > 64) return us;
        return std::max(us, 4.0 + (double)slices * (bm == 32 ? (slices < 128 ? 0.37 : 0.55) : slices < 128 ? 0.68 : 0.76));
    }
    const double small = 4.9;
    if (!is_staged(p.dtype, config_id) || us <= small) return us;
    const bool f32 = p.dtype == MMBO_F32, off_a = p.lda % (f32 ? 4 : 8) != 0, off_b = p.ldb % (f32 ? 4 : 8) != 0;
    const double a = f32 ? (p.transA ? 1.13 : 1.32) : (p.transA ? 1.35 : 1.65), b = f32 ? 1.05 : (p.transB ? 1.55 : 1.25);
    return small + (us - small) * (!f32 ? 2.15 : off_a || off_b ? 2.0 : 1.75) * (off_a ? a : 1.0) * (off_b ? b : 1.0);
}

// By 8 % at least: nearer than that the models do not tell the two apart (110 drawn shapes, against the tables' configs alone:
// 1.367 times faster in the geometric mean, two slower by over 2 %; without the margin 1.361 and seven).  Updates of a C inside a
// much larger matrix: by 17 %.  Neither model knows where the columns of C lie; of 13 such shapes modelled up to 1.2 times faster seven
// were slower (fp16 NT 512 x 797 x 96, ldc 44160, 5.1 -> 6.4 us), of 15 beyond that none.
// The ring kernel's 64 x 64 tile without a split, picked for a few microseconds of work, takes 2.65 us less than its model says (55 drawn
// shapes, 2.1 - 3.0), which matters only here: by 2.0 us, as this kernel takes 0.6 less on its smallest calls and 5 % less on the others.  us
// here / there: fp16 TT 1024 x 640 x 512 6.4 / 5.1, TT 4 x 576 x 320 x 512 8.4 / 5.7, TN 768 x 128 x 640 4.4 / 5.5, fp32 NN 448 x 768 x 304 7.0 / 8.1.
// Against a staged config the model of this kernel, too, is at the end of what it was fitted to: from 8 us on by a quarter (fp32) or a
// fifth, and by half where it says a wavefront per work-group on problems over 32 wide or, fp32, over 40 us (one wavefront to a work-group
// reuses what the staged kernel's four share), unless the tables' own model says so, too.  Drawn calls that left the staged kernel: with a
// margin of 8 % alone fp16 1.62 times faster in the geometric mean, 71 of 3,960 slower by over 3 %, fp32 1.30 and 168 of 2,120; with these
// bars fp16 1.66 and 24 of 2,816, fp32 (a third of them in planes) 1.47 and 6 of 191.  us, staged / split by wavefront: fp16 NT 191 x 102 x
// 32 x 512 43.0 / 12.6, 2 x 2267 x 7424 43.2 / 11.4, TT 12320 x 4 x 5569 91.7 / 22.8; the other way, fp32 TN 128 x 56 x 512 x 384 49.1 / 87.7.
WavePick pick_wave_over(const WaveShape &q, bool may_split, int config_id, double table_us)
{
    const double us = config_us(q, config_id, table_us);
    double bar = (q.wide_c ? 0.83 : 0.92) * us;
    if (q.dtype != MMBO_F64 && config_id == ring_config_id(3, 0)) bar = std::min(bar, us - 2.0);
    const WavePick w = pick_wave(q, may_split, bar);             // (none at `bar` or beyond)
    // fp64 against a slice's round trip (config_us): from 50 us on by a quarter.  Drawn calls that left the tables' kernel for it: 1.77 times faster in
    // the geometric mean and 93 of 3,675 slower by over 3 % with 8 % throughout, 1.90 and 3 of 1,381 so.  us: NT 409 x 456 x 18536 652.6 / 164.3.
    if (w.tile >= 0 && q.dtype == MMBO_F64 && w.us >= 50.0 && w.us >= (q.wide_c ? 0.83 : 0.92) * table_us && w.us >= 0.75 * us)
        return WavePick{-1, 0, 0, bar};
    // (fp32: nor for fewer runs of k than the config's, whose sums are the more exact -- 3 of 3,000 drawn calls, TT 55 x 4480 x 2298 eight runs, here four --
    // unless, again, the tables' own model says so)
    if (w.tile >= 0 && q.dtype == MMBO_F32 && is_staged(q.dtype, config_id) && w.us >= (q.wide_c ? 0.83 : 0.92) * table_us &&
        w.waves * w.split < config_ref(config_id).split)
        return WavePick{-1, 0, 0, bar};
    if (w.tile >= 0 && w.us >= 8.0 && is_staged(q.dtype, config_id)) {
        const bool half = (w.waves == 1 && std::min(q.m, q.n) > 32) || (q.dtype == MMBO_F32 && w.us > 40.0);
        if (w.us >= (q.wide_c ? 0.83 : 0.92) * table_us && w.us >= (q.dtype == MMBO_F32 ? (half ? 0.45 : 0.75) : half ? 0.5 : 0.8) * us) return WavePick{-1, 0, 0, bar};
    }
    return w;
}
WaveShape packed_shape(int dtype, int transA, int transB, size_t m, size_t n, size_t k, int batch, bool read_c)
{
    return wave_shape(dtype, transA, transB, m, n, k, batch, transA ? k : m, transB ? n : k, m, read_c);
}

// ---- fp32 on the bf16 pipes (gemm_planes.hpp) -----------------------------------------------------------------------------

// Modelled microseconds: work-groups run in rounds of 256, one to a CU; each costs a start and an epilogue (that reads C) and its slices
// (a group's, where several share k), which take less where part of the chip is idle -- the clock rises --, beside that what the bytes take
// from memory.  Constants: least squares over 12,600 times, 1,454 drawn shapes x every (tile, splits) that fits them: 5 - 7 % rms; the
// pick is 0.4 % behind the fastest of them on average, 22 % at worst.  (The 64 x 64 tile: 3,520 times of 2,142 shapes, 5 %.)
double planes_model_us(int tile, int split, size_t m, size_t n, size_t k, int batch)
{
    static const double start[NUM_PLANES_TILES] = {5.25 + 2.52, 3.65 + 1.61, 3.96 + 0.94, 3.98 + 0.44}, slice[NUM_PLANES_TILES] = {1.803, 1.090, 1.312, 1.251},
                        idle_chip[NUM_PLANES_TILES] = {0.848, 0.878, 0.886, 0.814};
    const double launch = 1.67, bytes_per_us = 4.04e6, hidden = 0.126, reduce = 2.88, reduce_per_mb = 0.320;
    const PlanesRow &r = kPlanesTiles[tile];
    const size_t slices = ceil_div(k, (size_t)kPlanesBk), per_split = ceil_div(slices, (size_t)split), splits = ceil_div(slices, per_split);
    const double wgs = (double)(ceil_div(m, (size_t)r.bm) * ceil_div(n, (size_t)r.bn) * splits) * batch;
    const double c_mb = (double)m * n * batch * 4e-6;
    auto round = [&](double busy) {
        return start[tile] + (double)ceil_div(per_split, (size_t)r.kg) * slice[tile] * (idle_chip[tile] + (1.0 - idle_chip[tile]) * busy);
    };
    const double full = std::floor(wgs / 256), last = wgs - full * 256;
    const double work = full * round(1.0) + (last > 0 ? round(last / 256) : 0.0);
    const double memory = (((double)m * k + (double)k * n) * batch * 4.0 + c_mb * 1e6) / bytes_per_us;
    return std::max(work, memory) + hidden * std::min(work, memory) + launch + (splits > 1 ? reduce + reduce_per_mb * c_mb * (double)splits : 0.0);
}

struct PlanesPick {
    int tile;           // row of kPlanesTiles; < 0: none
    int split;
};

// Are sums in planes, k added up in `runs` runs, as exact as those of the fp32 MFMAs in `others`?  The error of a sum grows with its runs' length; how
// much longer a run in planes may be depends on the operands.  Equal 2-norm errors against 64 bits, k = 512 .. 32768: uniform [-1, 1] and normal
// operands eight times as long, uniform [0, 1] 2.8 times, operands spread over 2^-10 .. 2^10 four times, over 2^-20 .. 2^20 of either sign twice (k = 512,
// 2048; 8192 1.9 times, 32768 1.5 times), positive ones twice from 256 k to a run on.  Shorter runs of the fp32 MFMAs leave planes less to gain -- the
// 32 products that one MFMA adds are cut to its largest one's bits --: k = 512 of positive operands over 2^-10 .. 2^10, fp32 MFMAs / planes, four runs of
// 128 1.4e-7 / 0.86e-7, eight of 64 0.89 / 0.85, sixteen of 32 0.78 / 0.91.  Of 300 drawn calls that come to planes, on four kinds of operands, none is
// less exact by over 0.1 %.  (Eight times throughout took 25 more of 3,000 drawn calls to planes and 16 into fewer splits: 1.18 times faster.)
bool planes_as_exact(size_t k, int runs, int others)
{
    if (others <= 1) return true;
    const size_t length = k / (size_t)others;
    return length >= 256 ? (k <= 4096 ? others <= 2 * runs : 2 * others <= 3 * runs) : length >= 128 && others <= runs;
}

// What the kernel is to run a shape with, where it beats what else would run it -- `us` microseconds modelled, k added up in `runs` runs -- by
// a tenth, from 16 us on by a twentieth (nearer than that the models do not tell them apart; the twentieth, and the ring kernel's model taken at
// its word from there on, moved 2,694 drawn calls, 1.16 times faster in the geometric mean; of 420 of that kind on the present kernel none is
// slower by over 2 %).  Partial sums (k split over work-groups) of at most max_bytes.
// Only where sums stay as exact (planes_as_exact); k below 64 was not measured to be on operands of widely different magnitudes.
// Not (planes_may_pay) for calls of a few microseconds, where a work-group has next to no slices to overlap anything with (us before / with it: TT 46 x 128 x
// 128 x 384 10.9 / 13.0, NT 1280 x 512 x 144 6.8 / 8.2; with fewer than five slices up to 30: NT 4334 x 1152 x 128 19.9 / 26.2, but of 40 us
// and more 1.13 - 1.2 times faster; NT 1735 x 652 x 160 11.2 / 13.2).
bool planes_may_pay(int transA, int transB, size_t m, size_t n, size_t k, double us)
{
    return k >= 64 && us >= (k < 160 ? 30.0 : k < 256 ? 16.0 : 12.0) && planes_shape_ok(transA, transB, m, n, k);
}
PlanesPick pick_planes(int transA, int transB, size_t m, size_t n, size_t k, int batch, int runs, double us, double max_bytes)
{
    PlanesPick best{-1, 0};
    double best_us = (us < 16.0 ? 0.90 : 0.95) * us;
    if (!planes_may_pay(transA, transB, m, n, k, us)) return best;
    for (int tile = 0; tile < NUM_PLANES_TILES; ++tile) {
        const PlanesRow &r = kPlanesTiles[tile];
        const size_t tiles = ceil_div(m, (size_t)r.bm) * ceil_div(n, (size_t)r.bn);
        for (int split : kSplits) {
            if ((size_t)batch * split > 65535) break;
            if (split > 1 && ((double)split * batch * (double)m * (double)n * sizeof(float) > max_bytes || tiles * batch * split > 1100 ||
                              k / kPlanesBk < (size_t)4 * r.kg * split))
                break;
            if (!planes_as_exact(k, split * r.kg, runs)) continue;
            const double t = planes_model_us(tile, split, m, n, k, batch);
            if (t < best_us) {
                best_us = t;
                best = PlanesPick{tile, split};
            }
        }
    }
    return best;
}

// ---- fp64 sums without a split over work-groups (gemm_dots.hpp) -------------------------------------------------------

// (a pair of rows that the edge cuts is the two that end there, so a row-contiguous operand has two at least)
bool dots_shape_ok(int tile, int transA, int transB, size_t m, size_t n, size_t k)
{
    const DotsRow &r = kDotsTiles[tile];
    return k > 0 && (transA || m >= 2) && (!transB || n >= 2) &&
           ceil_div(m, 4 * (size_t)r.fm) * ceil_div(n, 4 * (size_t)r.fn) <= 65535;
}
// (its tiles' own spans are smaller, but a call that no config of the tables may take is refused: what the smallest of them, 32 x 32, takes)
bool dots_span_ok(int transA, int transB, size_t lda, size_t ldb)
{
    return tile_span_ok(TileRow{32, 32, kDotsStep, 0, 0}, transA, transB, lda, ldb, sizeof(double));
}

// Modelled microseconds: work-groups run in rounds of 256, one to a CU; each costs a start and its steps, a step as long as the slowest of the
// lines its CU pulls, the lines all CUs pull, and its products; a wavefront's steps share round trips.  Beside that what the bytes take from
// memory, and C, which goes element by element.  Constants: least squares over 7,100 times, 1,192 drawn shapes x every tile: 12 % rms.
double dots_model_us(const WaveShape &p, int tile)
{
    const double launch = 1.62, start = 0.705, cu_bytes = 110.6e3, chip_bytes = 24.5e6, block = 0.0033, load = 0.0104, round_trips = 1.92 / 8,
                 memory_bytes = 7.64e6, hidden = 0.72, c_us = 37.7e-6;
    const DotsRow &r = kDotsTiles[tile];
    auto lines = [&](int rows, size_t dim, bool k_contiguous, size_t ld) {
        const double here = (double)std::min((size_t)rows, ceil_div(dim, (size_t)4) * 4);
        const bool on_lines = ld % 16 == 0;
        if (k_contiguous) return here * kDotsStep * 8 * (on_lines ? 1.0 : 1.25);
        return kDotsStep * (on_lines ? 128.0 : here * 8 + 112);
    };
    const double line_bytes = lines(4 * r.fm, p.m, p.transA, p.lda) + lines(4 * r.fn, p.n, !p.transB, p.ldb);
    const double steps = (double)p.k / kDotsStep, wgs = (double)(ceil_div(p.m, 4 * (size_t)r.fm) * ceil_div(p.n, 4 * (size_t)r.fn)) * p.batch;
    auto round = [&](double busy) {
        const double step = std::max(std::max(line_bytes / cu_bytes, line_bytes * busy / chip_bytes), r.fm * r.fn * block + (r.fm + r.fn) * load);
        return start + std::max(steps * step, round_trips * std::ceil(steps / kDotsWaves));
    };
    const double full = std::floor(wgs / 256), last = wgs - 256 * full, c = (double)p.m * p.n * p.batch;
    const double work = full * round(256) + (last > 0 ? round(last) : 0.0);
    const double memory = ((double)p.m * p.k + (double)p.k * p.n) * p.batch * 8 / memory_bytes + c * (p.read_c ? 16 : 8) / memory_bytes;
    return std::max(launch + std::max(work, memory) + hidden * std::min(work, memory) + c * c_us, 5.1);
}

// The row of kDotsTiles to run a shape on, where it beats the `us` microseconds modelled of what else would by a tenth, below 7 us and with two
// row-contiguous operands -- each line that their narrow tiles touch is partly others' -- by a sixth; -1: none.  (6,518 drawn fp64 shapes, with
// a tenth for all: taken for 645, which went 1.62 times faster in the geometric mean -- 2.1 - 2.6 with two k-contiguous operands,
// 1.1 - 1.4 with none --, 14 slower by over 3 %, eight of them with none and four more below 7 us.)
int pick_dots(const WaveShape &p, double us)
{
    int best = -1;
    double best_us = (us < 7.0 || (!p.transA && p.transB) ? 0.84 : 0.90) * us;
    for (int tile = 0; tile < NUM_DOTS_TILES; ++tile) {
        if (!dots_shape_ok(tile, p.transA, p.transB, p.m, p.n, p.k)) continue;
        const double t = dots_model_us(p, tile);
        if (t < best_us) {
            best_us = t;
            best = tile;
        }
    }
    return best;
}

// What the automatic pick runs for a shape.  The models are walked once per shape and thread (2 - 4 us, a part of what a
// small call takes); a small table of four ways keeps the answers, which are a function of the key alone.
// Whether a call needs a workspace, and how large a one at most, follows from the shape alone, not from beta or leading dimensions:
// a program runs a shape once and then captures a call of that shape that may differ in those, which cannot allocate.  So a
// shape whose pick of mmbo_select_config splits k is first planned with packed operands and without C.  Where that plan needs no
// workspace, no call of the shape does; where it needs one, every call of the shape holds one as large.
struct Plan {
    PlanesPick planes;  // tile < 0: dots
    int dots;           // row of kDotsTiles; < 0: wave
    WavePick wave;      // tile < 0: config_id
    int config_id;
    bool workspace;     // may partial sums go through memory?
    size_t reserve;     // bytes of workspace that a call sees to although it may need less itself
};

thread_local size_t g_plans_made = 0;

Plan plan_for(const WaveShape &p)
{
    struct Key {
        int dtype, transA, transB, batch, read_c, wide_c, lines_a, lines_b;
        size_t m, n, k;
    };
    struct Entry {
        bool used;
        Key key;
        Plan plan;
    };
    constexpr int kSets = 32, kWays = 4;
    struct Set {
        Entry way[kWays];
        unsigned next;              // the way that goes next: the oldest
    };
    static thread_local Set cache[kSets];
    const size_t per_line = 128 / (p.dtype == MMBO_F64 ? 8 : p.dtype == MMBO_F32 ? 4 : 2);
    Key key;
    std::memset(&key, 0, sizeof(key));                   // (compared as bytes)
    key.dtype = p.dtype; key.transA = p.transA; key.transB = p.transB; key.batch = p.batch; key.read_c = p.read_c; key.wide_c = p.wide_c;
    auto alignment = [&](size_t ld) { return ld % per_line == 0 ? 2 : ld % (per_line / 8) == 0; };
    key.lines_a = alignment(p.lda); key.lines_b = alignment(p.ldb);
    key.m = p.m; key.n = p.n; key.k = p.k;
    size_t h = p.m * 0x9E3779B97F4A7C15ull ^ p.n * 0xC2B2AE3D27D4EB4Full ^ p.k * 0x165667B19E3779F9ull ^
               (size_t)(p.batch * 16 + p.dtype * 4 + p.transA * 2 + p.transB) * 0x27D4EB2F165667C5ull;
    Set &set = cache[(h >> 32) % kSets];
    for (const Entry &e : set.way)
        if (e.used && std::memcmp(&e.key, &key, sizeof(key)) == 0) return e.plan;
    ++g_plans_made;
    Plan plan;
    double table_us;
    plan.config_id = select_config(p.dtype, p.transA, p.transB, p.m, p.n, p.k, p.batch, &table_us);
    const int table_split = p.dtype == MMBO_F64 ? 1 : config_ref(plan.config_id).split;
    auto choose = [&](const WaveShape &q, bool may_split) { return pick_wave_over(q, may_split, plan.config_id, table_us); };
    plan.workspace = false;
    plan.reserve = 0;
    const double table_bytes = (double)table_split * p.batch * p.m * p.n * sizeof(float);
    const WaveShape packed_call = packed_shape(p.dtype, p.transA, p.transB, p.m, p.n, p.k, p.batch, false);
    WavePick packed{-1, 0, 0, 0};
    if (table_split > 1) packed = choose(packed_call, true);
    if (table_split == 1) {
        plan.wave = choose(p, false);
    } else {
        plan.workspace = packed.tile < 0 || packed.split > 1;
        if (!plan.workspace) {
            plan.wave = pick_wave(p, false);
        } else {
            plan.wave = choose(p, true);
            if (packed.tile >= 0 && plan.wave.tile < 0 && table_bytes > (double)kWaveSumsBytes) plan.wave = pick_wave(p, true);
            plan.reserve = packed.tile < 0 ? (size_t)std::min(table_bytes, 1e18) : kWaveSumsBytes;
        }
    }
    // fp32 in planes: a matter of the shape alone, as its workspace is -- against what would run the packed call without C.
    plan.planes = PlanesPick{-1, 0};
    // (What would run it takes what the table's config does at most: small calls need not walk the models for that.)
    if (p.dtype == MMBO_F32 && !config_ref(plan.config_id).planes &&
        planes_may_pay(p.transA, p.transB, p.m, p.n, p.k, config_us(packed_call, plan.config_id, table_us))) {
        if (table_split == 1) packed = choose(packed_call, false);
        // (the ring kernel's 64 x 64 tile takes some 2 us less than its model says for a few microseconds of work: see pick_wave_over.  From 16
        // on it takes what the model says or more: 1024^3 21.4 - 22.3, modelled 21.6 - 22.2; in planes 19.2 - 19.8.)
        const double us = packed.tile >= 0 ? packed.us : plan.config_id == ring_config_id(3, 0) && table_us < 16.0 ? table_us - 2.0 : config_us(packed_call, plan.config_id, table_us);
        auto runs = [&](const WavePick &w) { return w.tile >= 0 ? w.waves * w.split : table_split; };
        plan.planes = pick_planes(p.transA, p.transB, p.m, p.n, p.k, p.batch, runs(packed), us,
                                  plan.workspace ? std::max(table_bytes, (double)kWaveSumsBytes) : 0.0);
        if (plan.planes.tile >= 0 && plan.planes.split > 1)
            plan.reserve = std::max(plan.reserve, (size_t)plan.planes.split * p.batch * p.m * p.n * sizeof(float));
        // (but a call whose beta or leading dimensions would have it run in more runs than the packed one without C keeps to those)
        if (plan.planes.tile >= 0 && !planes_as_exact(p.k, plan.planes.split * kPlanesTiles[plan.planes.tile].kg, runs(plan.wave))) plan.planes.tile = -1;
    }
    plan.dots = p.dtype == MMBO_F64 ? pick_dots(p, plan.wave.tile >= 0 ? plan.wave.us : config_us(p, plan.config_id, table_us)) : -1;
    set.way[set.next] = Entry{true, key, plan};
    set.next = (set.next + 1) % kWays;
    return plan;
}

// What MMBO_CONFIG_AUTO runs: the kernel on bf16 planes, that for small results of long sums or the split-by-wavefront kernel, which take any
// alignment, or a config.
struct Route {
    bool planes;
    PlanesPick planes_pick;
    bool dots;
    int dots_tile;
    bool wave;
    WavePick pick;
    int config_id;
    size_t reserve;     // of Plan
};

inline size_t element_size(int dtype) { return dtype == MMBO_F64 ? 8 : dtype == MMBO_F32 ? 4 : 2; }

// aligned16: A, B, their leading dimensions and batch strides are whole 16-byte groups.
int route_for(const WaveShape &p, bool aligned16, WsSource ws_source, Route &r)
{
    const size_t esz = element_size(p.dtype);
    const Plan plan = plan_for(p);
    r.pick = plan.wave;
    r.reserve = plan.reserve;
    r.planes_pick = plan.planes;
    r.planes = plan.planes.tile >= 0 && tile_span_ok(planes_tile(plan.planes.tile), p.transA, p.transB, p.lda, p.ldb, esz);
    if (ws_source == WsSource::kStatic && r.planes) {
        // partial sums that fit the array of the entry point that allocates nothing -- unless what else would run the call is more exact then
        auto fitting = [&](int split) {
            while (split > 1 && (double)split * p.batch * (double)p.m * (double)p.n * sizeof(float) > (double)kScratchPartialBytes) split /= 2;
            return split;
        };
        r.planes_pick.split = fitting(plan.planes.split);
        if (r.planes_pick.split < plan.planes.split)
            r.planes = planes_as_exact(p.k, r.planes_pick.split * kPlanesTiles[plan.planes.tile].kg,
                                       plan.wave.tile >= 0 ? plan.wave.waves * plan.wave.split : fitting(config_ref(plan.config_id).split));
    }
    r.dots_tile = plan.dots;
    r.dots = plan.dots >= 0 && dots_span_ok(p.transA, p.transB, p.lda, p.ldb);
    // (a pair of slices must span less than the 2 GiB of a buffer descriptor)
    r.wave = plan.wave.tile >= 0 &&
             tile_span_ok(TileRow{kWaveTiles[plan.wave.tile].bm, kWaveTiles[plan.wave.tile].bn, (int)(2 * 64 / esz), 0, 0}, p.transA, p.transB,
                          p.lda, p.ldb, esz);
    int id = r.config_id = plan.config_id;
    if (r.planes || r.dots || r.wave) return MMBO_OK;
    const bool f64 = p.dtype == MMBO_F64;
    // The pick is made from the shape alone.  The ring kernels also need 16-byte aligned A and B, every
    // direct-to-LDS kernel a tile's span of an operand below 2 GiB: where the operands at hand do not qualify, the
    // x16 config of the same tile and split (any alignment), or the staged kernel, takes the call.
    if (!f64 && !aligned16) {
        const ConfigRef c = config_ref(id);
        if (c.ring && !c.x16) {
            static const int x16_of_ring[NUM_RING_TILES] = {0, 2, 3, 4};
            int si = 0;
            while (si + 1 < NUM_SPLITS && kSplits[si] != c.split) ++si;
            const int tile = x16_of_ring[c.tile];
            id = ring_shape_ok(p.dtype, tile, c.split, p.transA, p.transB, p.m, p.n, p.k, true)
                     ? x16_config_id(tile, si) : select_staged(p.dtype, p.m, p.n, p.k, p.batch);
        }
    }
    // The entry point that allocates nothing holds kScratchPartialBytes of partial sums: where the pick's GlobalSplitU
    // needs more, the same tile runs with the largest split that fits (down to none), so that every shape still
    // runs under MMBO_CONFIG_AUTO.  (A config the caller names is taken as named, or refused.)  A shape planned without a workspace
    // whose leading dimensions are too large for that plan runs without a split.
    if (!f64 && (ws_source == WsSource::kStatic || !plan.workspace)) {
        const ConfigRef c = config_ref(id);
        int si = split_index(c.split);
        auto fits = [&](int sidx) {
            if (kSplits[sidx] == 1) return true;
            if (!plan.workspace) return false;
            if ((double)kSplits[sidx] * p.batch * (double)p.m * (double)p.n * sizeof(float) > (double)kScratchPartialBytes) return false;
            return c.planes || !c.ring || ring_shape_ok(p.dtype, c.tile, kSplits[sidx], p.transA, p.transB, p.m, p.n, p.k, c.x16);
        };
        while (si > 0 && !fits(si)) --si;
        id = c.planes ? planes_config_id(c.tile, si) : c.x16 ? x16_config_id(c.tile, si) : c.ring ? ring_config_id(c.tile, si) : staged_config_id(c.tile, si);
    }
    if (!tile_span_ok(config_tile(p.dtype, id), p.transA, p.transB, p.lda, p.ldb, esz)) {
        // enormous leading dimensions: the first staged tile (no split-K) whose span fits, large tiles first
        const int ntiles = f64 ? NUM_F64_TILES : NUM_TILES;
        id = -1;
        for (int tile = 0; tile < ntiles && id < 0; ++tile)
            if (tile_span_ok(config_tile(p.dtype, tile), p.transA, p.transB, p.lda, p.ldb, esz)) id = tile;
        if (id < 0) return MMBO_ERR_INVALID_SIZE;
    }
    r.config_id = id;
    return MMBO_OK;
}

// The partial sums' buffer of a call that needs `needed` bytes (0: none), in a.ws; a call of the library's own workspace sees to
// `reserve` bytes as well.
int hold_workspace(hipStream_t s, WsSource ws_source, size_t needed, size_t reserve, WsHold &hold, GemmArgs &a)
{
    size_t bytes = needed;
    if (ws_source == WsSource::kLibrary && reserve > (needed > 0 ? std::max(needed, kWaveSumsBytes) : 0)) {
        // (a call under capture takes what is there: it cannot allocate, nor must it where it needs nothing)
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone) bytes = std::max(bytes, reserve);
    }
    if (bytes == 0) return MMBO_OK;
    char *base = nullptr;
    const int rc = ws_source == WsSource::kStatic ? static_scratch(&base) : workspace(s, bytes, hold, &base);
    if (rc != MMBO_OK && needed > 0) return rc;
    a.ws = reinterpret_cast<float *>(base);
    return MMBO_OK;
}

// The split-by-wavefront kernel with the given pick on checked arguments; `a` holds the operands, sizes, strides and scalars.
int run_wave(const WaveShape &p, const WavePick &w, GemmArgs &a, hipStream_t s, WsSource ws_source, size_t reserve)
{
    const WaveRow &row = kWaveTiles[w.tile];
    const size_t esz = element_size(p.dtype), bk = 64 / esz;
    a.nwg0 = (uint32_t)ceil_div(p.m, row.bm); a.nwg1 = (uint32_t)ceil_div(p.n, row.bn);
    // (how tiles are laid over the XCDs: see the kernel)
    const bool tall = a.nwg0 >= a.nwg1;
    const size_t long_ld = tall ? p.lda : p.ldb, line = 128 / esz;
    const bool whole_lines = (tall ? !p.transA : p.transB) && long_ld % line == 0 && (uintptr_t)(tall ? a.A : a.B) % 128 == 0 &&
                             (tall ? row.bm : row.bn) % line == 0 && (tall ? a.nwg0 : a.nwg1) % 8 == 0;
    a.wgm = whole_lines ? 1 : 8;
    a.nxcd = whole_lines ? 1 : 8;
    a.columns_first = whole_lines && !tall && a.nwg0 > 1;
    const size_t pairs = ceil_div(ceil_div(p.k ? p.k : 1, bk), 2), pairs_per_split = ceil_div(pairs, (size_t)w.split);
    a.splits = (uint32_t)ceil_div(pairs, pairs_per_split);
    a.k_per_split = (uint32_t)(a.splits > 1 ? pairs_per_split * 2 * bk : (p.k ? p.k : 1));
    a.wave_pairs = (uint32_t)ceil_div(pairs_per_split, (size_t)w.waves);
    const uint32_t per16 = (uint32_t)(16 / esz);
    const uint32_t past_a = p.transA ? 0 : wave::columns_without_a_successor(a.m, per16, a.lda),
                   past_b = p.transB ? wave::columns_without_a_successor(a.n, per16, a.ldb) : 0;
    a.no_successor = past_a > past_b ? past_a : past_b;
    a.vec_c = ((uintptr_t)a.C % 16 == 0) && ((a.ldc * esz) % 16 == 0) && (((size_t)a.strideC * esz) % 16 == 0);
    WsHold ws_hold;
    const size_t needed = a.splits > 1 ? (size_t)a.splits * p.batch * p.m * p.n * sizeof(float) : 0;
    if (int rc = hold_workspace(s, ws_source, needed, reserve, ws_hold, a)) return rc;
    hipError_t e = p.dtype == MMBO_F64 ? dispatch_wave<2, 0>(w.tile, p.transA, p.transB, a, w.waves, s)
                   : p.dtype == MMBO_F32 ? dispatch_wave<0, 0>(w.tile, p.transA, p.transB, a, w.waves, s)
                                         : dispatch_wave<1, 0>(w.tile, p.transA, p.transB, a, w.waves, s);
    if (e != hipSuccess) return hip_fail(e);
    if (a.splits > 1) {
        e = launch_splitk_reduce(p.dtype, a, s);
        if (e != hipSuccess) return hip_fail(e);
    }
    return MMBO_OK;
}

// The fp64 kernel for small results of long sums on row `tile` of kDotsTiles.
int run_dots(const WaveShape &p, int tile, GemmArgs &a, hipStream_t s)
{
    const DotsRow &r = kDotsTiles[tile];
    a.nwg0 = (uint32_t)ceil_div(p.m, 4 * r.fm); a.nwg1 = (uint32_t)ceil_div(p.n, 4 * r.fn);
    a.columns_first = a.nwg1 > a.nwg0;
    const hipError_t e = dispatch_dots<0>(tile, p.transA, p.transB, a, s);
    return e == hipSuccess ? MMBO_OK : hip_fail(e);
}

// What both entry points and the queries check of a problem before anything else.
int check_problem(int dtype, int transA, int transB, size_t m, size_t n, size_t k, size_t lda, size_t ldb, size_t ldc, int batch)
{
    if (!valid_dtype(dtype)) return MMBO_ERR_INVALID_DTYPE;
    if ((transA & ~1) || (transB & ~1)) return MMBO_ERR_INVALID_OP;
    const size_t kMaxDim = 0x7FFFFFFFull;
    if (m > kMaxDim || n > kMaxDim || k > kMaxDim || lda > kMaxDim || ldb > kMaxDim || ldc > kMaxDim)
        return MMBO_ERR_INVALID_SIZE;
    if (batch < 0 || batch > 65535) return MMBO_ERR_INVALID_SIZE;
    // BLAS rule: a leading dimension is at least 1 and at least the operand's stored row count
    const size_t need_a = transA ? k : m, need_b = transB ? n : k;
    if (lda < (need_a ? need_a : 1) || ldb < (need_b ? need_b : 1) || ldc < (m ? m : 1)) return MMBO_ERR_INVALID_SIZE;
    return MMBO_OK;
}

int gemm_impl(int dtype, int transA, int transB, size_t m, size_t n, size_t k,
              const void *alpha, const void *A, size_t lda, long long strideA,
              const void *B, size_t ldb, long long strideB, const void *beta, void *C,
              size_t ldc, long long strideC, int batch, int config_id, void *stream, WsSource ws_source,
              const WavePick *named_wave = nullptr, const PlanesPick *named_planes = nullptr, const int *named_dots = nullptr)
{
    if (!valid_dtype(dtype)) return MMBO_ERR_INVALID_DTYPE;
    if ((transA & ~1) || (transB & ~1)) return MMBO_ERR_INVALID_OP;
    if (!alpha || !beta) return MMBO_ERR_NULL_POINTER;
    if (int rc = check_problem(dtype, transA, transB, m, n, k, lda, ldb, ldc, batch)) return rc;
    if (strideA < 0 || strideB < 0 || strideC < 0) return MMBO_ERR_INVALID_SIZE;
    if (config_id != MMBO_CONFIG_AUTO && (config_id < 0 || config_id >= mmbo_num_configs(dtype)))
        return MMBO_ERR_INVALID_CONFIG;
    if (m == 0 || n == 0 || batch == 0) return MMBO_OK;          // nothing to write
    if (!C) return MMBO_ERR_NULL_POINTER;
    if (k != 0 && (!A || !B)) return MMBO_ERR_NULL_POINTER;

    const bool f64 = dtype == MMBO_F64;
    const double alpha_d = f64 ? *static_cast<const double *>(alpha) : (double)*static_cast<const float *>(alpha);
    const double beta_d = f64 ? *static_cast<const double *>(beta) : (double)*static_cast<const float *>(beta);
    const float alpha_f = (float)alpha_d, beta_f = (float)beta_d;

    const size_t esz = element_size(dtype);
    GemmArgs a;
    std::memset(&a, 0, sizeof(a));
    a.A = A; a.B = B; a.C = C; a.ws = nullptr;
    a.alpha = alpha_f; a.beta = beta_f;
    a.alpha_d = alpha_d; a.beta_d = beta_d;
    a.m = (uint32_t)m; a.n = (uint32_t)n; a.k = (uint32_t)k;
    a.lda = (uint32_t)lda; a.ldb = (uint32_t)ldb; a.ldc = (uint32_t)ldc;
    a.strideA = strideA; a.strideB = strideB; a.strideC = strideC;
    a.batch = (uint32_t)batch;
    auto aligned16 = [&](const void *p, size_t ld, long long stride) {
        return ((uintptr_t)p % 16 == 0) && ((ld * esz) % 16 == 0) && (((size_t)stride * esz) % 16 == 0);
    };
    a.vec_a = aligned16(A, lda, strideA);
    a.vec_b = aligned16(B, ldb, strideB);
    hipStream_t s = static_cast<hipStream_t>(stream);

    PlanesPick planes{-1, 0};
    size_t reserve = 0;
    if (named_planes) {
        planes = *named_planes;
    } else if (config_id == MMBO_CONFIG_AUTO) {
        const WaveShape p = wave_shape(dtype, transA, transB, m, n, k, batch, lda, ldb, ldc, f64 ? beta_d != 0.0 : beta_f != 0.0f);
        if (named_wave) return run_wave(p, *named_wave, a, s, ws_source, 0);
        if (named_dots) return run_dots(p, *named_dots, a, s);
        Route r;
        if (int rc = route_for(p, a.vec_a && a.vec_b, ws_source, r)) return rc;
        if (r.planes) planes = r.planes_pick;
        else if (r.dots) return run_dots(p, r.dots_tile, a, s);
        else if (r.wave) return run_wave(p, r.pick, a, s, ws_source, r.reserve);
        config_id = r.config_id;
        if (dtype == MMBO_F32) reserve = r.reserve;
    }
    const ConfigRef cref = planes.tile >= 0 ? ConfigRef{false, planes.tile, planes.split, false, true}
                           : f64 ? ConfigRef{false, config_id, 1, false, false} : config_ref(config_id);
    int split = cref.split;
    const RingRow &rr = cref.x16 ? kX16Tiles[cref.tile] : kRingTiles[cref.ring ? cref.tile : 0];
    const TileRow r = cref.planes ? planes_tile(cref.tile) : config_tile(dtype, config_id);
    if (cref.planes && !planes_shape_ok(transA, transB, m, n, k)) return MMBO_ERR_INVALID_CONFIG;
    if (cref.ring && !ring_shape_ok(dtype, cref.tile, split, transA, transB, m, n, k, cref.x16)) return MMBO_ERR_INVALID_CONFIG;

    if (!tile_span_ok(r, transA, transB, lda, ldb, esz)) return MMBO_ERR_INVALID_CONFIG;

    size_t nwg0 = ceil_div(m, r.bm), nwg1 = ceil_div(n, r.bn);
    if (nwg0 * nwg1 > 0x7FFFFFFFull) return MMBO_ERR_INVALID_SIZE;
    // split-K: slices are whole stages; never more slices than stages
    size_t stages = ceil_div(k, r.bk);
    if (stages < 1) stages = 1;
    if ((size_t)split > stages) split = (int)stages;
    size_t k_per_split = ceil_div(stages, (size_t)split) * r.bk;
    split = (int)ceil_div(k ? k : 1, k_per_split);        // the last split takes what is left, a partial slice included
    if ((size_t)batch * split > 65535) return MMBO_ERR_INVALID_SIZE;

    a.nwg0 = (uint32_t)nwg0; a.nwg1 = (uint32_t)nwg1;
    a.wgm = 8;
    a.nxcd = 8;
    a.splits = (uint32_t)split;
    a.k_per_split = (uint32_t)(split > 1 ? k_per_split : (k ? k : 1));
    // (tiles that run one work-group per CU: 256 x 256 and 192 x 192)
    a.chip_block = cref.x16 && rr.depth * (rr.bm + rr.bn) * 64 > 80 * 1024 && nwg0 >= 16 && nwg1 >= 16;
    // batches of problems of at most 32 tiles (an XCD's CUs hold them at one time): each problem on one XCD
    a.batch_xcd = split == 1 && batch >= a.nxcd && batch % a.nxcd == 0 && nwg0 * nwg1 <= 32;
    auto on_lines = [&](const void *p, size_t ld, long long stride) {
        return ((uintptr_t)p % 128 == 0) && ((ld * esz) % 128 == 0) && (batch == 1 || ((size_t)stride * esz) % 128 == 0);
    };
    a.line_rows = on_lines(A, lda, strideA) && on_lines(B, ldb, strideB);
    a.quartered = f64 ? (uint32_t)quartered_tiles(cref.tile, nwg0 * nwg1, batch, k) : 0;
    a.ws_narrow = (size_t)r.bn * m * 4 < 0x7FFFFF00ull;
    a.vec_c = aligned16(C, ldc, strideC);
    // (the x16 kernel addresses C as a buffer with 32-bit offsets: where a tile's span of C, its columns x ldc, does not fit them, C goes
    // out element by element instead)
    a.c_narrow = (size_t)r.bn * ldc * esz < 0x7FFFFF00ull;
    // fp16: columns on odd elements, some or all of them, leave by the epilogue that keeps its accesses to whole groups of rows on
    // dwords (a group that the edge cuts is read and written where it lies).  NT 8192 x 2048 x 256, us: C on an odd element, ldc 8192,
    // 27.6 -> 21.6, with beta 39.1 -> 29.3; ldc 8193 29.6 -> 20.9 and 39.2 -> 30.2; from a dword 20.9 and 30.1.
    // (one split and a narrow C: the x16 kernel's variants for odd columns and for a prefetched old C take nothing else)
    a.c_odd = cref.x16 && dtype == MMBO_F16 && split == 1 && a.c_narrow && ((uintptr_t)C % 4 != 0 || ldc % 2 != 0 || (batch > 1 && strideC % 2 != 0));
    // beta != 0 on the x16 kernel's fp16 path: the old C of a tile is fetched into LDS under the tile's last slices (through
    // buffer loads, at any alignment)
    a.c_prefetch = cref.x16 && dtype == MMBO_F16 && beta_f != 0.0f && split == 1 && a.c_narrow && !a.c_odd;
    // C with the non-temporal hint: only where resident work-groups walk at least four rounds of tiles (256 CUs) with a long
    // slice loop -- there the operand panels the next tiles share are worth more in the L2 than a fast epilogue (8192^3:
    // +0.3 %); with fewer rounds or a short k plain stores win (fp16 6144^3 +1.6 %, 44160 x 2048 x 384 +2.7 %, 64 x 512^3 +14 %).
    // Columns off 16 bytes never: their pieces of lines have to meet in the L2 (NN 8192 x 8192 x 4096, C off by 4 bytes, us: fp16
    // 463 -> 411, fp32 off by 8 bytes 3,917 -> 3,799).
    a.c_stream = cref.x16 && a.vec_c && rr.depth * (rr.bm + rr.bn) * 64 > 80 * 1024 && (size_t)nwg0 * nwg1 >= 4 * 256 && k >= 4096;

    if (cref.ring && !cref.x16 && (!a.vec_a || !a.vec_b)) return MMBO_ERR_INVALID_CONFIG;
    // Split-K: the partial sums go to the stream's own workspace (or the static one), and both launches that use it (the
    // GEMM and the reduction, which adds the splits in a fixed order) are queued before the hold on that workspace
    // is given up.
    const size_t needed = split > 1 ? (size_t)split * batch * m * n * sizeof(float) : 0;
    if (ws_source == WsSource::kStatic && needed > kScratchPartialBytes) return MMBO_ERR_WORKSPACE;
    WsHold ws_hold;
    if (int rc = hold_workspace(s, ws_source, needed, reserve, ws_hold, a)) return rc;
    hipError_t e;
    if (f64) e = dispatch_dgemm<0>(cref.tile, transA, transB, a, s);
    else if (cref.planes) e = dispatch_planes<0>(cref.tile, transA, transB, a, s);
    else if (cref.x16) e = dtype == MMBO_F32 ? dispatch_x16<0, 0>(cref.tile, transA, transB, a, s)
                                        : dispatch_x16<1, 0>(cref.tile, transA, transB, a, s);
    else if (cref.ring) e = dtype == MMBO_F32 ? dispatch_ring<0, 0>(cref.tile, transA, transB, a, s)
                                         : dispatch_ring<1, 0>(cref.tile, transA, transB, a, s);
    else e = dtype == MMBO_F32 ? dispatch_tile<0, 0>(cref.tile, transA, transB, a, s)
                               : dispatch_tile<1, 0>(cref.tile, transA, transB, a, s);
    if (e != hipSuccess) return hip_fail(e);
    if (split > 1) {
        e = launch_splitk_reduce(dtype, a, s);
        if (e != hipSuccess) return hip_fail(e);
    }
    return MMBO_OK;
}

}  // namespace

extern "C" {

int mmbo_auto_info(int dtype, int transA, int transB, size_t m, size_t n, size_t k, size_t lda, size_t ldb, size_t ldc, int reads_c,
                   int batch, int *config_id, mmbo_config_desc *out)
{
    if (!config_id || !out) return MMBO_ERR_NULL_POINTER;
    if (int rc = check_problem(dtype, transA, transB, m, n, k, lda, ldb, ldc, batch)) return rc;
    Route r{};
    if (m != 0 && n != 0 && batch != 0) {
        const size_t esz = element_size(dtype);
        const bool aligned16 = (lda * esz) % 16 == 0 && (ldb * esz) % 16 == 0;
        if (int rc = route_for(wave_shape(dtype, transA, transB, m, n, k, batch, lda, ldb, ldc, reads_c != 0), aligned16, WsSource::kLibrary, r)) return rc;
    }
    if (r.planes) {
        const bool has_id = r.planes_pick.tile < kPlanesIdTiles;
        *config_id = has_id ? planes_config_id(r.planes_pick.tile, split_index(r.planes_pick.split)) : MMBO_CONFIG_AUTO;
        describe_planes(r.planes_pick.tile, r.planes_pick.split, out);
        return MMBO_OK;
    }
    if (r.dots) {
        const DotsRow &row = kDotsTiles[r.dots_tile];
        std::memset(out, 0, sizeof(*out));
        const int bm = 4 * row.fm, bn = 4 * row.fn;
        std::snprintf(out->name, sizeof(out->name), "MT%03dx%03dx%02d_WT%03dx%03d_W%d_GSU01_LSU%02d_DTL1_DOTS%d", bm, bn, kDotsStep, bm, bn,
                      kDotsWaves, kDotsWaves, row.depth);
        out->macro_tile_m = out->wave_tile_m = bm;
        out->macro_tile_n = out->wave_tile_n = bn;
        out->depth_u = kDotsStep;
        out->threads = kDotsWaves * 64;
        out->split_k = 1;
        out->lds_bytes = kDotsWaves * row.depth * (row.fm + row.fn) * 1024;
        *config_id = MMBO_CONFIG_AUTO;
        return MMBO_OK;
    }
    if (!r.wave) {
        *config_id = r.config_id;
        return mmbo_config_info(dtype, r.config_id, out);
    }
    const WaveRow &row = kWaveTiles[r.pick.tile];
    std::memset(out, 0, sizeof(*out));
    const int bk = (int)(64 / element_size(dtype));
    std::snprintf(out->name, sizeof(out->name), "MT%03dx%03dx%02d_WT%03dx%03d_W%d_GSU%02d_LSU%02d_DTL1_WAVE%d", row.bm, row.bn, bk, row.bm,
                  row.bn, r.pick.waves, r.pick.split, r.pick.waves, row.depth);
    out->macro_tile_m = out->wave_tile_m = row.bm;
    out->macro_tile_n = out->wave_tile_n = row.bn;
    out->depth_u = bk;
    out->threads = r.pick.waves * 64;
    out->split_k = r.pick.split;
    const int sum_size = dtype == MMBO_F64 ? 8 : 4, ring = row.depth * (row.bm + row.bn) * 64, partial = (row.bm + 16 / sum_size) * row.bn * sum_size;
    out->lds_bytes = r.pick.waves * std::max(ring, partial);
    *config_id = MMBO_CONFIG_AUTO;
    return MMBO_OK;
}

// Not part of the interface: how often this thread has walked the models for the automatic pick.
size_t mmbo_internal_plans_made(void) { return g_plans_made; }

// Not part of the interface: mmbo_gemm_strided_batched on a given row of kWaveTiles, with given wavefronts per work-group and
// GlobalSplitU, whatever the pick is -- the tests reach every instantiation of the kernel through it.
int mmbo_internal_wave_gemm(int dtype, int transA, int transB, size_t m, size_t n, size_t k,
                            const void *alpha, const void *A, size_t lda, long long strideA,
                            const void *B, size_t ldb, long long strideB, const void *beta, void *C,
                            size_t ldc, long long strideC, int batch, int tile, int waves, int split, void *stream)
{
    if (!valid_dtype(dtype)) return MMBO_ERR_INVALID_DTYPE;
    if (tile < 0 || tile >= wave_tiles(dtype) || (waves != 1 && waves != 4 && waves != 8) || waves > wave_max_waves(kWaveTiles[tile]) || split < 1 ||
        split > 64 || (dtype == MMBO_F64 && split > 1))
        return MMBO_ERR_INVALID_CONFIG;
    if (int rc = check_problem(dtype, transA, transB, m, n, k, lda, ldb, ldc, batch)) return rc;
    const size_t esz = element_size(dtype);
    const WaveRow &row = kWaveTiles[tile];
    if (k == 0 || ceil_div(m, row.bm) * ceil_div(n, row.bn) > 65535 ||
        !tile_span_ok(TileRow{row.bm, row.bn, (int)(2 * 64 / esz), 0, 0}, transA, transB, lda, ldb, esz))
        return MMBO_ERR_INVALID_SIZE;
    const WavePick pick{tile, waves, split, 0.0};
    return gemm_impl(dtype, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, batch,
                     MMBO_CONFIG_AUTO, stream, WsSource::kLibrary, &pick);
}

// Not part of the interface: mmbo_gemm_strided_batched (fp32) on a given row of kPlanesTiles with a given GlobalSplitU.
int mmbo_internal_planes_gemm(int transA, int transB, size_t m, size_t n, size_t k, const void *alpha, const void *A, size_t lda,
                              long long strideA, const void *B, size_t ldb, long long strideB, const void *beta, void *C, size_t ldc,
                              long long strideC, int batch, int tile, int split, void *stream)
{
    if (tile < 0 || tile >= NUM_PLANES_TILES || split < 1 || split > 16) return MMBO_ERR_INVALID_CONFIG;
    const PlanesPick pick{tile, split};
    return gemm_impl(MMBO_F32, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, batch,
                     MMBO_CONFIG_AUTO, stream, WsSource::kLibrary, nullptr, &pick);
}

// Not part of the interface: mmbo_gemm_strided_batched (fp64) on a given row of kDotsTiles.
int mmbo_internal_dots_gemm(int transA, int transB, size_t m, size_t n, size_t k, const void *alpha, const void *A, size_t lda,
                            long long strideA, const void *B, size_t ldb, long long strideB, const void *beta, void *C, size_t ldc,
                            long long strideC, int batch, int tile, void *stream)
{
    if (tile < 0 || tile >= NUM_DOTS_TILES) return MMBO_ERR_INVALID_CONFIG;
    if (int rc = check_problem(MMBO_F64, transA, transB, m, n, k, lda, ldb, ldc, batch)) return rc;
    if (!dots_shape_ok(tile, transA, transB, m, n, k) || !dots_span_ok(transA, transB, lda, ldb)) return MMBO_ERR_INVALID_SIZE;
    return gemm_impl(MMBO_F64, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, batch,
                     MMBO_CONFIG_AUTO, stream, WsSource::kLibrary, nullptr, nullptr, &tile);
}

int mmbo_gemm_strided_batched(int dtype, int transA, int transB, size_t m, size_t n, size_t k,
                              const void *alpha, const void *A, size_t lda, long long strideA,
                              const void *B, size_t ldb, long long strideB, const void *beta, void *C,
                              size_t ldc, long long strideC, int batch, int config_id, void *stream)
{
    return gemm_impl(dtype, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, batch,
                     config_id, stream, WsSource::kLibrary);
}

int mmbo_gemm_strided_batched_static_workspace(int dtype, int transA, int transB, size_t m, size_t n, size_t k,
                                               const void *alpha, const void *A, size_t lda, long long strideA,
                                               const void *B, size_t ldb, long long strideB, const void *beta, void *C,
                                               size_t ldc, long long strideC, int batch, int config_id, void *stream)
{
    return gemm_impl(dtype, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, batch,
                     config_id, stream, WsSource::kStatic);
}

int mmbo_gemm(int dtype, int transA, int transB, size_t m, size_t n, size_t k, const void *alpha,
              const void *A, size_t lda, const void *B, size_t ldb, const void *beta, void *C, size_t ldc,
              int config_id, void *stream)
{
    return mmbo_gemm_strided_batched(dtype, transA, transB, m, n, k, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc,
                                     0, 1, config_id, stream);
}

}  // extern "C"
