// fp64 kernel for small results of long sums: a few rows by a few columns of C, k of thousands.
//
// fp64 never splits k over work-groups (its partial sums have no place in memory), so the only work-groups there are come from C's
// tiles, and the smallest tile of the other kernels is 16 x 16: 49 x 45 x 57216 ran on 12 of the 256 CUs, each bound by its one or two round
// trips per slice.  Here a work-group has a tile of 4 x 4 up to 16 x 8, and what bounds it is the memory lines that its CU pulls through its
// vector path.  v_mfma_f64_4x4x4 multiplies four independent 4 x 4 x 4 blocks; all four are the same 4 x 4 block of C, on different k, so one
// instruction is 4 x 4 x 16 without a wasted product.  Which k a lane holds does not matter as long as it holds the same of A and B.
//
// A step is 32 k: lane l multiplies row (column) l % 4 of each block at k = 2 * (l / 4) + 0, 1.  Wavefronts take the steps in turn, each
// through a ring of its own in LDS that direct loads fill: no barrier before the sums, and a CU has up to 144 KB of requests in flight.
// (LDS only for the sake of the loads: requests whose lanes lie in the order of memory.  Straight to registers, four lanes of an
// instruction in four rows of a k-contiguous operand, a CU got 37 - 50 bytes a ns, here 90 - 110.)  The blocks' sums, then the wavefronts', are added
// in a fixed order.  Rows past the edge repeat the last ones (their sums are not stored); the last k % 32 go by elements that exist.
//
// us, split-by-wavefront kernel / here: 49 x 45 x 57216 TN 174.1 / 41.6, TT 215.4 / 93.2, NN 214.8 / 99.0, NT 255.1 / 144.6 (of a row-contiguous
// operand every k is a line of its own: 128 bytes for 32); TN 128 x 128 x 20576 70.4 / 33.3, 128 x 32 x 7023 26.1 / 7.9; against the
// staged kernel, TN 3963 x 56 x 8081 309.6 / 204.4.
#pragma once

#include "gemm_ring.hpp"

namespace mmbo {

namespace dots {

constexpr int kStep = 32;

// One operand's part of a step: F blocks of four rows (columns), F KB, a direct load each.
//   k-contiguous: block after block, row after row of 256 bytes; 16-byte chunk c of row i of a block sits at c ^ 4 * i, so that the four
//   rows' chunks that a fragment read takes lie in different banks.
//   row-contiguous, a pair of blocks: 64 bytes (rows 2 * i + 0, 1 for block 0, 1 of the pair) of every even k, then of every odd one.
//   row-contiguous, one block: 32 bytes of every k.
template <bool KC, int F>
struct Operand {
    static_assert(F == 1 || F % 2 == 0, "one block or pairs");
    static constexpr bool PAIRS = !KC && F > 1;

    // byte offset of what lane l of load f fetches, from the tile's first row (row-contiguous: from 8 bytes in front of it) at the
    // step's first k
    __device__ static inline uint32_t load_offset(int lane, int f, uint32_t ld, uint32_t here)
    {
        if constexpr (KC) {
            const uint32_t i = lane >> 4, chunk = (lane & 15) ^ (i << 2);
            return min(f * 4 + i, here - 1) * ld * 8 + chunk * 16;
        } else if constexpr (PAIRS) {
            const int r = (f & ~1) * 4 + 2 * (lane & 3);
            return (2 * (lane >> 2) + (f & 1)) * ld * 8 + (uint32_t)(min(r, (int)here - 2) + 1) * 8;
        } else {
            return (lane >> 1) * ld * 8 + (uint32_t)(min(2 * (lane & 1), (int)here - 2) + 1) * 8;
        }
    }
    __device__ static inline uint32_t row(uint32_t i, int f) { return PAIRS ? (f & ~1) * 4 + 2 * i + (f & 1) : f * 4 + i; }

    // x[f][t]: lane l's row of block f at its k number t.  A pair of rows that the edge cuts came as the two that end there.
    __device__ static inline void read(double (&x)[F][2], const char *part, int lane, uint32_t here)
    {
        const uint32_t i = lane & 3, q = lane >> 2;
        if constexpr (KC) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const f64x2 v = *reinterpret_cast<const f64x2 *>(part + f * 1024 + i * 256 + ((q ^ (i << 2)) << 4));
                x[f][0] = v[0];
                x[f][1] = v[1];
            }
        } else if constexpr (PAIRS) {
#pragma unroll
            for (int f = 0; f < F; f += 2)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f64x2 v = *reinterpret_cast<const f64x2 *>(part + (f + t) * 1024 + lane * 16);
                    x[f][t] = v[0];
                    x[f + 1][t] = v[1];
                }
            if (here % 2 != 0) {
#pragma unroll
                for (int f = 0; f < F; f += 2) {
                    const bool cut = f * 4 + 2 * i + 1 == here;
#pragma unroll
                    for (int t = 0; t < 2; ++t) x[f][t] = cut ? x[f + 1][t] : x[f][t];
                }
            }
        } else {
            const uint32_t slot = here % 2 != 0 && i + 1 == here ? i + 1 : i;
#pragma unroll
            for (int t = 0; t < 2; ++t) x[0][t] = *reinterpret_cast<const double *>(part + (2 * q + t) * 32 + slot * 8);
        }
    }
    // the last k_here < 32 of k, straight from memory
    __device__ static inline void read_tail(double (&x)[F][2], const char *step, uint32_t ld, uint32_t here, uint32_t k_here, int lane)
    {
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t r = min(row(lane & 3, f), here - 1), k = 2 * (lane >> 2) + t;
                x[f][t] = 0.0;
                if (k < k_here) x[f][t] = *reinterpret_cast<const double *>(step + (KC ? (size_t)r * ld + k : (size_t)k * ld + r) * 8);
            }
    }
};

}  // namespace dots

template <int FM, int FN, int WAVES, int DEPTH>
struct DotsCfg {
    static constexpr int STEP_BYTES = (FM + FN) * 1024, RING_BYTES = DEPTH * STEP_BYTES, LDS_BYTES = WAVES * RING_BYTES;
    static constexpr int SUMS = FM * FN * 16;             // of a wavefront
    static_assert((DEPTH - 1) * (FM + FN) < 64, "vmcnt counts to 63");
    static_assert(SUMS <= WAVES * 64 && SUMS * 8 <= RING_BYTES, "a thread for every element of C; partial sums fit the rings");
};

template <bool TA, bool TB, int FM, int FN, int WAVES, int DEPTH>
__global__ void __launch_bounds__(WAVES * 64)
gemm_dots_kernel(const GemmArgs args)
{
    using namespace dots;
    using Cfg = DotsCfg<FM, FN, WAVES, DEPTH>;
    constexpr int BM = 4 * FM, BN = 4 * FN, LOADS = FM + FN;
    using OpA = Operand<TA, FM>;
    using OpB = Operand<!TB, FN>;

    extern __shared__ __attribute__((aligned(1024))) char lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t batch = blockIdx.x;

    // A single problem's tiles are regrouped so that each XCD has a contiguous run of them, longer side first: it reads its part of the
    // longer operand and all of the shorter one.
    uint32_t tile = blockIdx.y;
    if (args.batch == 1) {
        const uint32_t x = tile & 7, each = gridDim.y >> 3, more = gridDim.y & 7;
        tile = x * each + min(x, more) + (tile >> 3);
    }
    uint32_t wg0, wg1;
    if (args.columns_first) {
        wg1 = __builtin_amdgcn_readfirstlane(tile / args.nwg0);
        wg0 = tile - wg1 * args.nwg0;
    } else {
        wg0 = __builtin_amdgcn_readfirstlane(tile / args.nwg1);
        wg1 = tile - wg0 * args.nwg1;
    }
    const uint32_t row0 = wg0 * BM, col0 = wg1 * BN;
    const uint32_t m_here = min((uint32_t)BM, args.m - row0), n_here = min((uint32_t)BN, args.n - col0);
    const uint32_t lda = args.lda, ldb = args.ldb;

    const char *gA = static_cast<const char *>(args.A) + ((int64_t)batch * args.strideA + (TA ? (int64_t)row0 * lda : (int64_t)row0)) * 8;
    const char *gB = static_cast<const char *>(args.B) + ((int64_t)batch * args.strideB + (TB ? (int64_t)col0 : (int64_t)col0 * ldb)) * 8;
    const int64_t stepA = (TA ? (int64_t)kStep : (int64_t)kStep * lda) * 8, stepB = (TB ? (int64_t)kStep * ldb : (int64_t)kStep) * 8;

    const int steps = args.k / kStep;
    const int count = steps > wave ? (steps - wave + WAVES - 1) / WAVES : 0;         // of this wavefront: wave, wave + WAVES, ..
    uint32_t offA[FM], offB[FN];
#pragma unroll
    for (int f = 0; f < FM; ++f) offA[f] = OpA::load_offset(lane, f, lda, m_here);
#pragma unroll
    for (int f = 0; f < FN; ++f) offB[f] = OpB::load_offset(lane, f, ldb, n_here);
    u32x4 curA = ring::slice_cursor(ring::uniform_address(gA + wave * stepA - (TA ? 0 : 8))),
          curB = ring::slice_cursor(ring::uniform_address(gB + wave * stepB - (TB ? 8 : 0)));
    char *const my_ring = lds + wave * Cfg::RING_BYTES;
    const uint32_t ring_base = (uint32_t)(uintptr_t)MMBO_LDS_PTR(my_ring);
    auto request = [&](int slot) {
        const uint32_t dst = ring_base + slot * Cfg::STEP_BYTES;
        ring::static_for<FM>([&](auto I) { ring::direct_load16<false>(curA, 0, offA[I], dst + I * 1024); });
        ring::static_for<FN>([&](auto I) { ring::direct_load16<false>(curB, 0, offB[I], dst + (FM + I) * 1024); });
        ring::advance(curA, WAVES * (uint64_t)stepA);
        ring::advance(curB, WAVES * (uint64_t)stepB);
    };

    // Old C of the element that this thread stores, ahead of everything else
    const uint32_t my_row = threadIdx.x % BM, my_col = threadIdx.x / BM;
    const bool stores = my_row < m_here && my_col < n_here;
    double *const c = static_cast<double *>(args.C) + (int64_t)batch * args.strideC + (int64_t)((size_t)(col0 + my_col) * args.ldc) + row0 + my_row;
    double old_c = 0.0;
    if (args.beta_d != 0.0 && stores) old_c = *c;

    double acc[2][FM][FN] = {};
    auto products = [&](const double (&a)[FM][2], const double (&b)[FN][2]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[t][i][j] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[i][t], b[j][t], acc[t][i][j], 0, 0, 0);
    };
    double a[FM][2], b[FN][2];
    auto read = [&](int slot) {
        OpA::read(a, my_ring + slot * Cfg::STEP_BYTES, lane, m_here);
        OpB::read(b, my_ring + slot * Cfg::STEP_BYTES + FM * 1024, lane, n_here);
    };
#pragma unroll
    for (int s = 0; s < DEPTH; ++s)
        if (s < count) request(s);
    // (the direct loads are asm statements that the compiler's own counting does not see; the "memory" clobbers keep the LDS reads
    // between them in order)
    int slot = 0, s = 0;
    for (; s + DEPTH < count; ++s) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * LOADS) : "memory");
        read(slot);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                         // in registers: the slot is free
        request(slot);
        products(a, b);
        slot = slot + 1 == DEPTH ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    for (; s < count; ++s) {
        read(slot);
        products(a, b);
        slot = slot + 1 == DEPTH ? 0 : slot + 1;
    }
    if (args.k % kStep != 0 && wave == steps % WAVES) {                             // (one with the shortest run)
        OpA::read_tail(a, gA + steps * stepA, lda, m_here, args.k % kStep, lane);
        OpB::read_tail(b, gB + steps * stepB, ldb, n_here, args.k % kStep, lane);
        products(a, b);
    }

    // lane l: row l / 16, column l % 4 of block l / 4 % 4
    __syncthreads();
    double *const partial = reinterpret_cast<double *>(lds);                       // [wavefront][block][16]
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            double s = acc[0][i][j] + acc[1][i][j];
            s += __shfl_xor(s, 4);
            s += __shfl_xor(s, 8);
            if ((lane & 12) == 0) partial[wave * Cfg::SUMS + (i * FN + j) * 16 + (lane >> 4) * 4 + (lane & 3)] = s;
        }
    __syncthreads();
    if (!stores) return;
    auto place = [](bool pairs, uint32_t r, uint32_t &block, uint32_t &i) {        // row(i, block) == r
        block = pairs ? (r >> 3) * 2 + (r & 1) : r >> 2;
        i = pairs ? (r >> 1) & 3 : r & 3;
    };
    uint32_t bi, i, bj, j;
    place(OpA::PAIRS, my_row, bi, i);
    place(OpB::PAIRS, my_col, bj, j);
    double sums[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) sums[w] = partial[w * Cfg::SUMS + (bi * FN + bj) * 16 + i * 4 + j];
    double sum = sums[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += sums[w];
    double v = args.alpha_d * sum;
    if (args.beta_d != 0.0) v = __builtin_fma(args.beta_d, old_c, v);
    *c = v;
}

}  // namespace mmbo
