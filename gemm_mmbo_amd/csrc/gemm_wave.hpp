// Kernel for problems that a round of shared-LDS tiles cannot spread over the chip: one or both of m and n small against
// the 256 CUs' worth of tiles, k long enough to split.
//
// Every wavefront of a work-group owns the same BM x BN tile of C and a run of k of its own (the reference's LocalSplitU,
// src/gemm/ref/vega20_Cijk_Ailk_Bjlk_DB.yaml solution fields); the partial tiles meet in LDS once, at the end, and are added in
// wavefront order, so the result does not depend on timing.  Nothing is shared before that: each wavefront fills a ring
// of LDS slices of its own with direct loads and waits for them by count, so there is no barrier in the loop, and a
// CU has up to 160 KB of requests in flight from its first microsecond on.  What bounds
// such a problem otherwise is a chain of round trips: dispatch, slice after slice at one memory latency each, partial
// sums through memory, a second dispatch to add them.
//
// Slices are 64 bytes per row as in gemm_x16.hpp; two at a time are requested and multiplied (the two halves of a
// 128-byte line of a k-contiguous operand back to back).
//
// Ragged problems: a k-contiguous operand repeats its last row for the rows past the edge.  A row-contiguous one reads
// whole 16-byte groups of rows; a group that straddles the edge takes in what follows in memory -- padding rows, the next
// column -- whose products land in rows and columns of the tile that are never stored.  Only the last few columns of
// the operand have nothing behind them: those (and a last partial slice) go through registers, a group that an edge cuts as
// the 16 bytes that end there.  So any m, n, k, leading dimension and element alignment is taken, and no byte outside the
// operands is read.
#pragma once

#include "gemm_ring.hpp"

namespace mmbo {

namespace wave {

// One operand's part of one slice: R rows x 64 bytes of k, fetched and read by one wavefront.
template <typename T, bool KC, int R>
struct Tile {
    static constexpr int ESZ = sizeof(T);
    static constexpr uint32_t EPC = 16 / ESZ;                     // elements per 16-byte group
    static constexpr int BYTES = R * 64;
    static constexpr int LOADS = R / 16;                          // direct loads (1 KB each) per slice
    static constexpr int F = R / 16;                              // 16-row MFMA blocks
    static constexpr int ROW_BYTES = R * ESZ;                     // row-contiguous: one k-row
    static constexpr int CPR = ROW_BYTES / 16;
    static constexpr int KPI = 1024 / ROW_BYTES;                  // k-rows per direct load
    static_assert(R == 16 || R == 32 || R == 64, "rows of a wavefront's tile");

    __device__ static inline uint32_t kc_off(uint32_t row, uint32_t chunk) { return row * 64 + ((chunk ^ ((row >> 1) & 3)) << 4); }
    // XOR on the chunk index that spreads the k-rows of one fragment read over the banks, as far as a k-row has chunks
    __device__ static inline uint32_t rc_mask(uint32_t k)
    {
        uint32_t x;
        if constexpr (ESZ == 8) x = ((k >> 1) & 1) << 3;
        else if constexpr (ESZ == 4) x = ((k >> 2) & 3) << 2;
        else if constexpr (R == 64) x = (((k >> 1) & 1) << 2) | (((k >> 3) & 1) << 1);
        else x = ((k >> 3) & 1) << 1;
        return x & (CPR - 1);
    }
    __device__ static inline uint32_t rc_off(uint32_t k, uint32_t chunk) { return k * ROW_BYTES + ((chunk ^ rc_mask(k)) << 4); }

    // byte offset, from the operand's origin at this slice, of what direct load i puts into LDS slot i * 64 + lane
    __device__ static inline uint32_t load_goff(int lane, int i, uint32_t ld, uint32_t valid)
    {
        if constexpr (KC) {
            const uint32_t row = i * 16 + (lane >> 2), chunk = (lane & 3) ^ ((row >> 1) & 3);
            return min(row, valid - 1) * ld * ESZ + chunk * 16;
        } else {
            const uint32_t k = i * KPI + lane / CPR, chunk = (lane % CPR) ^ rc_mask(k);
            return k * ld * ESZ + min(chunk, (valid - 1) / EPC) * 16;
        }
    }

    // The same slots through registers: k_here (<= the slice) columns of k exist, `valid` rows; only elements that exist are
    // read, those past k are zero (rows past the edge only feed rows of the tile that are never stored).  `before`: how many
    // elements of the contiguous dimension lie in front of this slice (k-contiguous: the k before it, else the rows).  A group
    // that the end of that dimension cuts comes as the 16 bytes that end there, shifted: element by element it was up to seven
    // memory round trips one behind the other, each waited for before the next (fp16 halves share registers).  fp16 TN, us: 33 x
    // 4096 x 4093 17.7 -> 15.1, 40 x 2048 x 1001 with beta 6.1 -> 5.8.  What does not exist is not requested, and nothing is
    // shifted where no group is cut (every line repeated and every group shifted, us: fp32 NT 480 x 1280 x 111 6.74 -> 6.41, 640 x 414 x
    // 1009 12.67 -> 12.53, fp16 NN 2269 x 25 x 744 4.80 -> 4.63, with beta 4.99 -> 4.83).
    __device__ static inline void fetch(u32x4 (&x)[LOADS], const char *g, uint32_t ld, uint32_t valid, uint32_t k_here, uint32_t before, int lane)
    {
        const uint32_t here = KC ? k_here : valid;                    // elements of the contiguous dimension from this slice's origin on
        if (__builtin_amdgcn_readfirstlane(before + here) < EPC) {    // the whole operand is shorter than 16 bytes in it
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                uint32_t line, first;
                slot(lane, i, line, first);
                union { T e[EPC]; u32x4 v; } u;
                const T *const p = reinterpret_cast<const T *>(g) + (size_t)(min(line, (KC ? valid : k_here) - 1) * ld);
#pragma unroll
                for (uint32_t e = 0; e < EPC; ++e) u.e[e] = p[min(first + e, here - 1)];
                const uint32_t kept = !KC && line >= k_here ? 0 : here - min(first, here);
#pragma unroll
                for (uint32_t e = 0; e < EPC; ++e)
                    if (e >= kept) u.e[e] = (T)0;
                x[i] = u.v;
            }
            return;
        }
        // (as a buffer from 16 bytes in front of the slice on: a request behind its 2 GiB returns zeros without going to memory)
        const __amdgpu_buffer_rsrc_t slice = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(ring::uniform_address(g - 16)), 0, 0x7fffffff, 0x00020000);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            uint32_t line, first;
            slot(lane, i, line, first);
            const uint32_t at = 16 + (KC ? min(line, valid - 1) : line) * ld * ESZ + min((int)first, (int)here - (int)EPC) * ESZ;
            x[i] = __builtin_amdgcn_raw_buffer_load_b128(slice, (KC ? first : line) >= k_here ? 0x80000000u : at, 0, 0);   // (element alignment is enough)
        }
    }
    // line (row of a k-contiguous tile, else k) and first element of LDS slot i * 64 + lane
    __device__ static inline void slot(int lane, int i, uint32_t &line, uint32_t &first)
    {
        if constexpr (KC) {
            line = i * 16 + (lane >> 2);
            first = ((lane & 3) ^ ((line >> 1) & 3)) * EPC;
        } else {
            line = i * KPI + lane / CPR;
            first = ((lane % CPR) ^ rc_mask(line)) * EPC;
        }
    }
    // What fetch requested, to LDS.  (The shift is here, behind both operands' requests: it is the first to wait for them.)
    __device__ static inline void put(u32x4 (&x)[LOADS], uint32_t valid, uint32_t k_here, uint32_t before, char *dst, int lane)
    {
        const uint32_t here = __builtin_amdgcn_readfirstlane(KC ? k_here : valid);
        if (here % EPC != 0 && __builtin_amdgcn_readfirstlane(before) + here >= EPC) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                uint32_t line, first;
                slot(lane, i, line, first);
                x[i] = ring::drop_elements<ESZ>(x[i], (int)first - min((int)first, (int)here - (int)EPC));
            }
        }
#pragma unroll
        for (int i = 0; i < LOADS; ++i) *reinterpret_cast<u32x4 *>(dst + i * 1024 + lane * 16) = x[i];
    }

    // Fragments of the F blocks for one slice.  fp16: lane l holds row l % 16, k = 8 * (l / 16) + 0..7 (one 16x16x32 MFMA).
    // fp32: k = 4 * (l / 16) + t in register t (four 16x16x4 MFMAs); fp64: k = 2 * (l / 16) + t (two 16x16x4 MFMAs).
    __device__ static inline void read(u32x4 (&x)[F], const char *lds, int lane)
    {
        const uint32_t r = lane & 15, g = lane >> 4;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            if constexpr (KC) {
                x[f] = *reinterpret_cast<const u32x4 *>(lds + kc_off(f * 16 + r, g));
            } else if constexpr (ESZ == 8) {
                union { double d[2]; u32x4 v; } u;
                const uint32_t m = f * 16 + r;
#pragma unroll
                for (int t = 0; t < 2; ++t) u.d[t] = *reinterpret_cast<const double *>(lds + rc_off(2 * g + t, m >> 1) + (m & 1) * 8);
                x[f] = u.v;
            } else if constexpr (ESZ == 4) {
                const uint32_t m = f * 16 + r;
#pragma unroll
                for (int t = 0; t < 4; ++t) x[f][t] = *reinterpret_cast<const uint32_t *>(lds + rc_off(4 * g + t, m >> 2) + (m & 3) * 4);
            } else {
                // transposing read: lane j of a 16-lane group points at k-row j/4, rows 4*(j%4)..+3, and receives row j of
                // the four k-rows
                const uint32_t j = r, m = f * 16 + (j & 3) * 4;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4 *)MMBO_LDS_PTR(
                        lds + rc_off(8 * g + 4 * h + (j >> 2), m >> 3) + (m & 7) * 2));
                    const u32x2 w = __builtin_bit_cast(u32x2, v);
                    x[f][2 * h] = w[0];
                    x[f][2 * h + 1] = w[1];
                }
            }
        }
    }
};

template <typename T> struct Acc { using block = f32x4; using elem = float; };
template <> struct Acc<double> { using block = f64x4; using elem = double; };

template <typename T>
__device__ inline void multiply(typename Acc<T>::block &c, const u32x4 &a, const u32x4 &b)
{
    if constexpr (sizeof(T) == 2) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    } else if constexpr (sizeof(T) == 4) {
        const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int t = 0; t < 4; ++t) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], y[t], c, 0, 0, 0);
    } else {
        const f64x2 x = __builtin_bit_cast(f64x2, a), y = __builtin_bit_cast(f64x2, b);
#pragma unroll
        for (int t = 0; t < 2; ++t) c = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], y[t], c, 0, 0, 0);
    }
}

// Columns at the end of a row-contiguous operand (`rows` of it, `per_group` elements to 16 bytes) whose last group of rows
// has no memory behind it.
inline uint32_t columns_without_a_successor(uint32_t rows, uint32_t per_group, uint32_t ld)
{
    const uint32_t past = (per_group - rows % per_group) % per_group;
    return (past + ld - 1) / ld;
}

}  // namespace wave

template <typename T, bool TA, bool TB, int BM, int BN, int DEPTH>
struct WaveCfg {
    using TileA = wave::Tile<T, TA, BM>;
    using TileB = wave::Tile<T, !TB, BN>;
    static constexpr int ESZ = sizeof(T);
    static constexpr int BK = 64 / ESZ;
    static constexpr int FM = BM / 16, FN = BN / 16;
    static constexpr int SLICE_BYTES = TileA::BYTES + TileB::BYTES;
    static constexpr int RING_BYTES = DEPTH * SLICE_BYTES;                       // per wavefront
    static constexpr int LOADS = TileA::LOADS + TileB::LOADS;                    // direct loads per slice
    static_assert(DEPTH % 2 == 0 && DEPTH * LOADS < 64, "slices go in pairs; vmcnt counts to 63");
    using elem = typename wave::Acc<T>::elem;
    static constexpr int GROUP = 16 / (int)sizeof(elem);                         // rows a thread adds up and stores at a time
    static constexpr int LDR = BM + GROUP;                                       // column stride of a partial tile in LDS
    static constexpr int PARTIAL_BYTES = LDR * BN * (int)sizeof(elem);
    static constexpr int lds_bytes(int waves)
    {
        return waves * (RING_BYTES > PARTIAL_BYTES ? RING_BYTES : PARTIAL_BYTES);
    }
};

template <typename T, bool TA, bool TB, int BM, int BN, int DEPTH, int MAX_WAVES>
__global__ void __launch_bounds__(MAX_WAVES * 64)
gemm_wave_kernel(const GemmArgs args)
{
    using namespace wave;
    using Cfg = WaveCfg<T, TA, TB, BM, BN, DEPTH>;
    using TileA = typename Cfg::TileA;
    using TileB = typename Cfg::TileB;
    using elem = typename Cfg::elem;
    constexpr int ESZ = Cfg::ESZ, BK = Cfg::BK, FM = Cfg::FM, FN = Cfg::FN, LOADS = Cfg::LOADS, GROUP = Cfg::GROUP, LDR = Cfg::LDR;

    extern __shared__ __attribute__((aligned(1024))) char lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int threads = blockDim.x, waves = threads >> 6;

    // Grid: (batch, tile, split), the batch index fastest: with a multiple of 8 problems the dispatcher's round-robin puts all
    // tiles of one problem on one XCD.  A single problem's work-groups are regrouped so that each XCD owns a contiguous run of
    // them, walked in blocks eight tile columns wide (wg_remap): it then reads few panels of either operand, and neighbours
    // share in one L2 the memory lines their edges cut through.  Against the dispatcher's own order, us: fp16 9150 x 2 x 5504 NT
    // 36.7 -> 26.9, 23711 x 793 x 352 NT 123.7 -> 69.4, fp64 1152 x 2156 x 1416 equal.  Not where the longer operand's rows lie on
    // memory lines and its tiles are whole lines wide (the host sets nxcd = 1): there is no line to share, and eight neighbours
    // on one XCD are 1 KB of every column, a few of its L2's channels; the dispatcher's order, longer side first, gives an XCD
    // every eighth tile of it (4096 x 128 x 4096 fp16 14.9 -> 12.9, 8192 x 64 x 2048 11.0 -> 8.8).  (Tile rows and columns are counted only
    // where there is more than one of both: each division is a hundred clocks or more on the way to the first request.)
    const uint32_t batch = blockIdx.x;
    uint32_t tile = blockIdx.y, split = blockIdx.z;
    if (args.batch == 1 && args.nxcd > 1) {
        const uint32_t total = gridDim.y * gridDim.z, id = tile + gridDim.y * split, x = id & 7, each = total >> 3, more = total & 7;
        tile = x * each + min(x, more) + (id >> 3);                                  // the first `more` XCDs have one more
        if (gridDim.z > 1) {
            split = __builtin_amdgcn_readfirstlane(tile / gridDim.y);
            tile -= split * gridDim.y;
        }
    }
    uint32_t wg0 = tile, wg1 = 0;
    if (args.nwg0 == 1) {
        wg0 = 0;
        wg1 = tile;
    } else if (args.columns_first) {
        wg0 = __builtin_amdgcn_readfirstlane(tile / args.nwg1);
        wg1 = tile - wg0 * args.nwg1;
    } else if (args.nwg1 != 1) {
        wg_remap(tile, args.nwg0, args.nwg1, args.wgm, 1, wg0, wg1);
        wg0 = __builtin_amdgcn_readfirstlane(wg0);
        wg1 = __builtin_amdgcn_readfirstlane(wg1);
    }
    const uint32_t row0 = wg0 * BM, col0 = wg1 * BN;
    const uint32_t m_here = min((uint32_t)BM, args.m - row0), n_here = min((uint32_t)BN, args.n - col0);
    const uint32_t lda = args.lda, ldb = args.ldb;
    const uint32_t k_begin = split * args.k_per_split;
    const uint32_t k_end = min(args.k, k_begin + args.k_per_split);

    const char *gA = static_cast<const char *>(args.A) +
                     ((int64_t)batch * args.strideA + (TA ? (int64_t)row0 * lda + k_begin : (int64_t)k_begin * lda + row0)) * ESZ;
    const char *gB = static_cast<const char *>(args.B) +
                     ((int64_t)batch * args.strideB + (TB ? (int64_t)k_begin * ldb + col0 : (int64_t)col0 * ldb + k_begin)) * ESZ;
    const int64_t stepA = (TA ? (int64_t)BK : (int64_t)BK * lda) * ESZ, stepB = (TB ? (int64_t)BK * ldb : (int64_t)BK) * ESZ;

    // whole slices that direct loads may fetch; the columns behind them (fewer than two slices) go through registers
    const bool edge = (!TA && m_here < (uint32_t)BM) || (TB && n_here < (uint32_t)BN);
    const uint32_t k_direct = edge ? min(k_end, args.k - min(args.k, args.no_successor)) : k_end;
    const int n_slice = __builtin_amdgcn_readfirstlane(k_direct > k_begin ? (int)((k_direct - k_begin) / BK) : 0);
    // a run of slices per wavefront, whole pairs
    const int run = 2 * (int)args.wave_pairs;
    const int first = min(run * wave, n_slice), count = min(run, n_slice - first);

    uint32_t offA[TileA::LOADS], offB[TileB::LOADS];
#pragma unroll
    for (int i = 0; i < TileA::LOADS; ++i) offA[i] = TileA::load_goff(lane, i, lda, m_here);
#pragma unroll
    for (int i = 0; i < TileB::LOADS; ++i) offB[i] = TileB::load_goff(lane, i, ldb, n_here);
    u32x4 curA = ring::slice_cursor(ring::uniform_address(gA + first * stepA)), curB = ring::slice_cursor(ring::uniform_address(gB + first * stepB));
    const uint32_t stepA32 = (uint32_t)stepA, stepB32 = (uint32_t)stepB;
    char *const my_ring = lds + wave * Cfg::RING_BYTES;
    const uint32_t ring_base = (uint32_t)(uintptr_t)MMBO_LDS_PTR(my_ring);

    // slices q and q + 1 of this wavefront's run into ring slots q % DEPTH and the next (q is even)
    auto request_pair = [&](int q, int slot) {
        const uint32_t dst = ring_base + slot * Cfg::SLICE_BYTES;
        if (q + 1 < count) {
            ring::static_for<TileA::LOADS>([&](auto I) {
                ring::direct_load16<false>(curA, stepA32, offA[I], dst + I * 1024);
                ring::direct_load16<true>(curA, stepA32, offA[I], dst + Cfg::SLICE_BYTES + I * 1024);
            });
            ring::static_for<TileB::LOADS>([&](auto I) {
                ring::direct_load16<false>(curB, stepB32, offB[I], dst + TileA::BYTES + I * 1024);
                ring::direct_load16<true>(curB, stepB32, offB[I], dst + Cfg::SLICE_BYTES + TileA::BYTES + I * 1024);
            });
        } else if (q < count) {
            ring::static_for<TileA::LOADS>([&](auto I) { ring::direct_load16<false>(curA, stepA32, offA[I], dst + I * 1024); });
            ring::static_for<TileB::LOADS>([&](auto I) { ring::direct_load16<false>(curB, stepB32, offB[I], dst + TileA::BYTES + I * 1024); });
        }
        ring::advance(curA, 2 * (uint64_t)stepA);
        ring::advance(curB, 2 * (uint64_t)stepB);
    };

    // Old C of the groups of rows this thread will store, requested ahead of everything else.
    T *const C = static_cast<T *>(args.C) + (int64_t)batch * args.strideC + (int64_t)col0 * args.ldc + row0;
    const bool to_ws = sizeof(T) < 8 && args.splits > 1;
    const bool read_c = !to_ws && (sizeof(T) == 8 ? args.beta_d != 0.0 : args.beta != 0.0f);
    constexpr int GPC = BM / GROUP, GROUPS = GPC * BN;                             // groups per column, per tile
    constexpr int AHEAD = GROUPS / 64 < 8 ? GROUPS / 64 : 8;                       // groups of a thread requested together
    struct rows_t { T e[GROUP]; };
    // (kept as they come, in whole registers: halves taken apart on arrival made every group wait for its own load, the first ones
    // ahead of the ring's first request.  A group that the edge cuts is the GROUP rows that end there, shifted where it is used -- the rows
    // in front of it may belong to another work-group, and are dropped.  fp16 with beta, us: TN 32 x 9356 x 1808 11.9 -> 11.3,
    // TT 619 x 523 x 389 on the device 6.6 -> 5.9.)
    typedef uint32_t raw_t __attribute__((ext_vector_type(GROUP * ESZ / 4)));
    raw_t old_c[AHEAD];
    static_assert(GROUPS % 64 == 0, "a wavefront's groups of one request are all in the tile or all behind it");
    auto request_c = [&](uint32_t first) {
        if (args.m >= (uint32_t)GROUP) {
#pragma unroll
            for (int a = 0; a < AHEAD; ++a) {
                const uint32_t g = first + a * threads;                            // (columns that do not exist repeat one that does)
                if (__builtin_amdgcn_readfirstlane(g) >= n_here * GPC) continue;    // (a wavefront with none of the columns only queues for nothing)
                const int r = min((int)((g % GPC) * GROUP), (int)m_here - GROUP);
                __builtin_memcpy(&old_c[a], C + (int64_t)((size_t)min(g / GPC, n_here - 1) * args.ldc) + r, sizeof(raw_t));
            }
        } else {
#pragma unroll
            for (int a = 0; a < AHEAD; ++a) {
                const uint32_t g = first + a * threads, r = (g % GPC) * GROUP, c = min(g / GPC, n_here - 1);
                if (__builtin_amdgcn_readfirstlane(g) >= n_here * GPC) continue;
                rows_t o;
#pragma unroll
                for (int e = 0; e < GROUP; ++e) o.e[e] = C[(size_t)c * args.ldc + min(r + e, m_here - 1)];
                old_c[a] = __builtin_bit_cast(raw_t, o);
            }
        }
    };
    auto old_rows = [&](const raw_t &x, uint32_t r) {
        const int past = args.m >= (uint32_t)GROUP ? (int)r - min((int)r, (int)m_here - GROUP) : 0;          // < GROUP where r is a row
        if constexpr (sizeof(raw_t) == 8) {
            const uint64_t v = __builtin_bit_cast(uint64_t, x) >> ((past & 3) * 16);
            return __builtin_bit_cast(rows_t, v);
        } else {
            if (m_here % GROUP == 0) return __builtin_bit_cast(rows_t, x);                                   // (no group is cut)
            return __builtin_bit_cast(rows_t, ring::drop_elements<ESZ>(x, past));
        }
    };
    if (read_c) request_c(tid);

    typename Acc<T>::block acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = typename Acc<T>::block{0, 0, 0, 0};
    auto multiply_slice = [&](const char *slice) {
        u32x4 a[FM], b[FN];
        TileA::read(a, slice, lane);
        TileB::read(b, slice + TileA::BYTES, lane);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) multiply<T>(acc[i][j], a[i], b[j]);
    };

    // Loads return in order: with DEPTH / 2 pairs requested, the oldest has landed when at most the others' loads are open.
    // (The LDS reads are ordinary loads: the direct loads are asm statements that the compiler's own counting does not
    // see, and the "memory" clobbers keep both sides in order.  Reading a pair ahead of the one being multiplied, into a
    // second register set, measured 0-6 % slower: the registers cost more wavefronts than the reads cost time.)
    constexpr int PAIRS = DEPTH / 2;
#pragma unroll
    for (int q = 0; q < DEPTH; q += 2) request_pair(q, q);
    int slot = 0, s = 0;
    for (; s + DEPTH + 1 < count; s += 2) {                                        // (a whole pair is left to request)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (PAIRS - 1) * LOADS) : "memory");
        multiply_slice(my_ring + slot * Cfg::SLICE_BYTES);
        multiply_slice(my_ring + (slot + 1) * Cfg::SLICE_BYTES);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                         // both slices are in registers: the slots are free
        request_pair(s + DEPTH, slot);
        slot = slot + 2 == DEPTH ? 0 : slot + 2;
    }
    for (; s < count; s += 2) {
        const int last = min((count + 1) / 2, s / 2 + PAIRS), behind = last - s / 2 - 1;        // pairs requested so far, and after this one
        const bool half = 2 * last > count;                                        // the last of them is one slice
        bool waited = false;
        ring::static_for<PAIRS - 1>([&](auto P) {
            constexpr int q = PAIRS - 1 - decltype(P)::value;
            if (!waited && behind == q) {
                if (half) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((2 * q - 1) * LOADS) : "memory");
                else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * q * LOADS) : "memory");
                waited = true;
            }
        });
        if (!waited) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        multiply_slice(my_ring + slot * Cfg::SLICE_BYTES);
        if (s + 1 < count) multiply_slice(my_ring + (slot + 1) * Cfg::SLICE_BYTES);
        if (s + DEPTH < count) {                                                   // (an odd run's last slice)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            request_pair(s + DEPTH, slot);
        }
        slot = slot + 2 == DEPTH ? 0 : slot + 2;
    }
    // What is left of k, at most two partial slices, on the wavefronts with the shortest runs.  (Requested ahead of the ring or
    // right behind it, to save the round trip: 0 - 1 % slower over 450 shapes.)
    for (uint32_t k0 = k_begin + n_slice * BK, w = waves - 1; k0 < k_end; k0 += BK, w = w == 0 ? waves - 1 : w - 1) {
        if (w != (uint32_t)wave) continue;
        const int64_t slices = (k0 - k_begin) / BK;
        const uint32_t k_here = min((uint32_t)BK, k_end - k0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                         // (the ring slot's last reads are done)
        u32x4 xa[TileA::LOADS], xb[TileB::LOADS];
        TileA::fetch(xa, gA + slices * stepA, lda, m_here, k_here, TA ? k0 : row0, lane);
        TileB::fetch(xb, gB + slices * stepB, ldb, n_here, k_here, TB ? col0 : k0, lane);
        TileA::put(xa, m_here, k_here, TA ? k0 : row0, my_ring, lane);
        TileB::put(xb, n_here, k_here, TB ? col0 : k0, my_ring + TileA::BYTES, lane);
        // (what a lane reads is what others of its wavefront wrote: in order for the hardware, but not something the compiler
        // can tell, which sees one thread's addresses)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        multiply_slice(my_ring);
    }

    // Partial tiles to LDS, column by column.  fp32 accumulators: lane l has rows 4 * (l / 16) .. +3 of column l % 16 of a
    // block; fp64: rows 4 * e + l / 16.
    __syncthreads();
    elem *const mine = reinterpret_cast<elem *>(lds + wave * Cfg::PARTIAL_BYTES);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            elem *p = mine + (j * 16 + (lane & 15)) * LDR + i * 16;
            if constexpr (sizeof(T) == 8) {
#pragma unroll
                for (int e = 0; e < 4; ++e) p[4 * e + (lane >> 4)] = acc[i][j][e];
            } else {
                *reinterpret_cast<f32x4 *>(p + 4 * (lane >> 4)) = acc[i][j];
            }
        }
    __syncthreads();

    typedef elem sums_t __attribute__((ext_vector_type(GROUP)));
    auto add_up = [&](uint32_t r, uint32_t c) {
        const char *p = lds + (c * LDR + r) * sizeof(elem);
        auto of = [&](int w) { return *reinterpret_cast<const sums_t *>(p + w * Cfg::PARTIAL_BYTES); };
        // All reads ahead of the additions, whose order stays: a loop over `waves` is one LDS round trip per wavefront (the
        // compiler unrolls it by eight and takes these seven in what is left over).  fp16 16 x 4096 x 4096: 8.45 -> 8.20 us.
        sums_t s = of(0);
        if (waves > 1) {                                         // 4 or 8
            const sums_t s1 = of(1), s2 = of(2), s3 = of(3);
            if (MAX_WAVES == 8 && waves == 8) {
                const sums_t s4 = of(4), s5 = of(5), s6 = of(6), s7 = of(7);
                return ((((((s + s1) + s2) + s3) + s4) + s5) + s6) + s7;
            }
            s = ((s + s1) + s2) + s3;
        }
        return s;
    };
    const elem alpha = sizeof(T) == 8 ? (elem)args.alpha_d : (elem)args.alpha, beta = sizeof(T) == 8 ? (elem)args.beta_d : (elem)args.beta;
    auto finish = [&](uint32_t g, const raw_t &old) {
        const uint32_t r = (g % GPC) * GROUP, c = g / GPC;
        if (c >= n_here || r >= m_here) return;
        const sums_t s = add_up(r, c);
        const bool whole = r + GROUP <= m_here;
        if (to_ws) {                                             // (never fp64)
            float *ws = args.ws + ((size_t)split * args.batch + batch) * (size_t)args.m * args.n + (size_t)(col0 + c) * args.m + row0 + r;
            if (whole) {
                __builtin_memcpy(ws, &s, sizeof(s));
            } else {
#pragma unroll
                for (int e = 0; e < GROUP; ++e)
                    if (r + e < m_here) ws[e] = (float)s[e];
            }
            return;
        }
        T *p = C + (size_t)c * args.ldc + r;
        rows_t o = read_c ? old_rows(old, r) : rows_t{};
#pragma unroll
        for (int e = 0; e < GROUP; ++e) {
            elem v = alpha * s[e];
            if (read_c) v = sizeof(T) == 8 ? (elem)__builtin_fma((double)beta, (double)o.e[e], (double)v)
                                           : (elem)__builtin_fmaf((float)beta, (float)o.e[e], (float)v);
            o.e[e] = (T)v;
        }
        if (whole) {
            __builtin_memcpy(p, &o, sizeof(rows_t));
        } else {
#pragma unroll
            for (int e = 0; e < GROUP; ++e)
                if (r + e < m_here) p[e] = o.e[e];
        }
    };
    for (uint32_t first = tid; first < GROUPS; first += AHEAD * threads) {
        if (read_c && first != (uint32_t)tid) request_c(first);
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
            if (first + a * threads < GROUPS) finish(first + a * threads, old_c[a]);
    }
}

}  // namespace mmbo
