// fp32 GEMM on the bf16 matrix pipes, without giving up a bit of the operands: every fp32 element is taken apart into three
// bf16 planes, x = x1 + x2 + x3 exactly (8 + 8 + 8 bits of significand, each rounded to nearest, so |x2| <= 2^-8 |x| and |x3| <= 2^-16 |x|),
// and the product of two elements is the sum of the six plane products that reach its 24 bits:
//     x*y = x1*y1 + (x1*y2 + x2*y1) + (x1*y3 + x3*y1 + x2*y2)           left out: x2*y3 + x3*y2 + x3*y3, below 2^-23 x*y, 2^-26 typically
// v_mfma_f32_16x16x32_bf16 forms products exactly and adds 32 of them at a time into fp32; x1*y1 goes to one accumulator, the five
// small products to another, and the two are added when the sum over k is whole.
//
// Why: an fp32 MFMA does 128 multiply-adds per clock and CU, a bf16 one 2,048, a sixth of that is 341.  us, before / with it (before: the fp32 MFMA
// kernels), NT 4096^3 with alpha and beta 948 / 538, TN 640 x 384 x 10000 accumulated 48.8 / 36.7, NN 2048^3 127 / 84, 4096 x 128 x 4096 39 / 32, NT 44160
// x 2048 x 384 accumulated 561 / 412.  What bounds it: at 4096^3 power -- 1.53 PFLOP/s of bf16 products at a 1.9 GHz clock, where a loop of nothing but
// these MFMAs sustains 1.9 on such data --, on smaller tiles the vector instructions that take the elements apart (64 x 64 tile with two
// groups of wavefronts, 1024^3, 21.0 us: without them and the LDS writes 15.1, without the MFMAs 16.3).
// Precision: fewer roundings than the fp32 MFMAs' (one per eight k instead of one per k), and those of the small products
// 2^-8 times smaller.  2-norm error against 64 bits, this form / v_mfma_f32_16x16x4_f32, uniform [-1, 1]: k = 64 4.5e-8 / 1.4e-7, 1024
// 1.7e-7 / 5.7e-7, 32768 1.2e-6 / 3.3e-6; uniform [0, 1] at 32768 8.5e-7 / 2.4e-6; operands spread over 2^-20 .. 2^20 at 64 6.1e-8 / 7.2e-8, at
// 32768 1.1e-6 / 1.4e-6.  (Six products into one accumulator: equal to the fp32 MFMAs', and behind them on spread operands.)  Sums of few terms that are
// not zero, uniform: 256 of 256 0.81e-7 / 2.87e-7, 16 3.1e-8 / 7.4e-8, two 2.58e-8 / 3.08e-8, but one 2.52e-8 / 2.48e-8: the products left out put 4 %
// of such sums one unit off the rounded product, by 1.61 half units at most.  (With x2*y3 and x3*y2 as well 2.48e-8, and NT 4096^3 557 -> 661 us, NN 1024^3 18.7
// -> 20.9, TN 640 x 384 x 10000 38.1 -> 41.0.)
//
// What the planes cannot hold is found out and computed again, for the whole tile, with fp32 MFMAs: see `again`.
//
// Structure, one work-group of eight (64 x 64 tile: twelve) wavefronts per BM x BN tile of C, two (three) to a SIMD (with one, the MFMAs' 16 clocks and the four of each other
// instruction add up: NN 4096^3 620 us instead of 557):
//   - slices of 32 k go memory -> registers (fp32) -> three planes -> LDS -> MFMA fragments.  Each element is taken apart once
//     per work-group (12 vector instructions per two elements), not once per wavefront that uses it.  The planes are written
//     k-contiguous whatever the operand's layout in memory (a lane that loaded rows instead of k holds them transposed in its registers),
//     so all four transposes run one loop of 128-bit fragment reads.  (The remainder below a plane by v_dot2_f32_bf16, which needs no
//     unpacking: fewer instructions, but they run in the matrix pipe, an MFMA and one of them 32 clocks.)
//   - LDS holds two slices: while slice s is multiplied, slice s + 1 is taken apart and written, and slice s + 2 is requested into the
//     registers that this frees, a slice's MFMAs ahead of its use.  (Two slices ahead, in a second set of registers: 1.2 % slower in the
//     128 x 128 tile, 2.9 in the 128 x 64, 2.5 in the 64 x 64, 4,243 drawn calls, most on short k; four: 2 - 5 % more.)  One barrier per slice.  The MFMAs of a slice's last row of blocks are issued behind the barrier, over the
//     first fragment reads of the next slice.
//   - every MFMA is followed by its share of the other instructions, in source order and fenced: left to the scheduler, MFMAs gather
//     and the vector unit idles, then the other way round.
//   - the 128 x 64 tile's two groups of wavefronts take every second slice each: 64 x 32 wavefront tiles read less LDS per MFMA than 32 x 32.
//     The 64 x 64 tile has three groups, three wavefronts to a SIMD: with two the barrier and the trips to LDS left the pipes idle for
//     part of each slice (two groups with four slices in flight each / three with two, before it was one, us: NN 1024^3 22.4 / 21.2, TN 1024^3 19.0 / 18.1, NN 768 x
//     1024 x 2048 31.5 / 30.0, TN 640 x 384 x 10000 128.1 / 114.8, with k split four ways 45.3 / 42.4; over 2,142 drawn shapes 1.08 -
//     1.13 times faster from 80 slices on, 1.02 - 1.05 from 12 on, below that 0.96 - 1.03).
//   - rows of a tile lie in LDS in the order 0, 4, 8, .., 1, 5, 9, ..: a lane's four accumulators of blocks BM/4 rows apart are then four
//     consecutive rows of C, sixteen lanes 256 contiguous bytes, and a lane's writes of four loaded rows fall on different banks.
#pragma once

#include <type_traits>

#include "gemm_ring.hpp"

namespace mmbo {
namespace planes {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

using ring::static_for;

constexpr int BK = 32;      // k per slice: one MFMA's, 64 bytes of a row in each plane

// 16-byte chunk c of row p of a plane lies at chunk c ^ swizzle(p).  Conflict-free for the 128-bit fragment reads (lane -> row l % 16,
// chunk l / 16; the hardware serves lanes 0-3, 12-15, 20-23, 24-27 and so on together) and for 8- and 16-byte writes of 16 consecutive rows.
__device__ inline uint32_t swizzle(uint32_t p) { return ((p >> 1) & 3) ^ (((p >> 3) & 1) * 3); }

// One operand's share of a slice: R rows x 32 k, NT threads, NV 16-byte loads each.
//   KC = true  (memory contiguous along k): load v of a thread is 4 k of one row; eight lanes take a row's 128 bytes.
//   KC = false (contiguous along the rows): a thread owns four consecutive rows x KU k, one load per k; eight lanes take 128 bytes of a k.
// "Physical" row p, the order in LDS, is row 4 * (p % (R/4)) + p / (R/4) of the tile.
template <bool KC, int R, int NT>
struct Operand {
    static constexpr bool K_CONTIGUOUS = KC;
    static constexpr int NV = R * 8 / NT;           // loads per thread and slice
    static constexpr int KU = NV;                   // (KC = false) k per thread
    static constexpr int PAIRS = NV * 2;            // pairs of elements a thread takes apart
    static constexpr int WORDS = KC ? 2 : KU / 2;   // 32-bit words (pairs) of one LDS write
    static constexpr int Q = R / 4;
    static constexpr int PLANE = R * 64;            // bytes
    static_assert(NV == 2 || NV == 4 || NV == 8, "2, 4 or 8 loads per thread");

    uint32_t voff[NV];          // byte offset of load v from the slice's origin (KC = true: from 16 bytes ahead of it)
    uint32_t wbase;             // LDS byte address of write 0 in plane 0
    uint32_t k_first;           // first k of this thread within the slice

    // the first row of quad q of a tile with `rows` rows: moved up where the tile ends inside it (KC = false)
    __device__ static inline int quad_row(int q, int rows) { return KC ? 4 * q : min(4 * q, rows - 4); }
    // rows a quad may start before the tile: then the origin lies that many rows up
    __device__ static inline int lead(int rows) { return !KC && rows < 4 ? 4 - rows : 0; }

    __device__ inline void init(uint32_t tid, uint32_t ld, int rows)
    {
        if constexpr (KC) {
            const uint32_t u = tid & 7, p0 = tid >> 3;
            k_first = u * 4;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const uint32_t p = v * (NT / 8) + p0, r = min(4 * (p % Q) + p / Q, (uint32_t)rows - 1);
                voff[v] = (r * ld + k_first + 4) * 4;
            }
            wbase = p0 * 64 + (((u >> 1) ^ swizzle(p0)) << 4) + (u & 1) * 8;
        } else {
            // lanes: eight quads, then the parts of a chunk of 8 k (the lanes of one pass of an LDS write, 128 bytes, then fall on different
            // banks), the other quads, the chunks
            constexpr uint32_t SUBS = 8 / KU;
            const uint32_t sub = (tid >> 3) % SUBS, rest = (tid >> 3) / SUBS, q = (tid & 7) | (rest % (Q / 8) << 3), c = rest / (Q / 8);
            k_first = c * 8 + sub * KU;
            const uint32_t r0 = (uint32_t)(quad_row(q, rows) + lead(rows));
#pragma unroll
            for (int v = 0; v < NV; ++v) voff[v] = ((k_first + v) * ld + r0) * 4;
            wbase = q * 64 + ((c ^ swizzle(q)) << 4) + sub * KU * 2;
        }
    }

    // bytes: 0 drops the request (zeros arrive)
    __device__ static inline u32x4 load(const char *origin, uint32_t off, int bytes)
    {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(origin), 0, bytes, 0x00020000);
        return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    }

    // From here on the requests are those of a slice of which only the first `left` (1 .. 31) k exist: every address inside the operand
    // (which has 4 k or more; the origin of a later slice has k ahead of it).  `fix_partial` puts the elements where they belong and
    // zeros behind them.
    __device__ inline void aim_partial(uint32_t ld, int left)
    {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            if constexpr (KC) voff[v] += (uint32_t)(min((int)k_first, left - 4) - (int)k_first) * 4;     // may begin up to 3 k before the slice
            else voff[v] -= (k_first + v - min(k_first + v, (uint32_t)left - 1)) * ld * 4;
        }
    }
    __device__ inline void fix_partial(u32x4 (&x)[NV], int left) const
    {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            if constexpr (KC) {
                const int here = left - (int)k_first;              // k of this group that exist
                const u32x4 t = x[v];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t y = 0;
                    // a cut group holds its `here` k at its end
                    if (here >= 4) y = t[e];
                    if (e < 3 && here == 3) y = t[(e + 1) & 3];
                    if (e < 2 && here == 2) y = t[(e + 2) & 3];
                    if (e < 1 && here == 1) y = t[3];
                    x[v][e] = y;
                }
            } else {
                if ((int)k_first + v >= left) x[v] = u32x4{0, 0, 0, 0};
            }
        }
    }
    // the two elements of pair x
    __device__ static inline uint32_t first_of(const u32x4 (&raw)[NV], int x)
    {
        if constexpr (KC) return raw[x / 2][2 * (x % 2)];
        else return raw[2 * (x % WORDS)][x / WORDS];
    }
    __device__ static inline uint32_t second_of(const u32x4 (&raw)[NV], int x)
    {
        if constexpr (KC) return raw[x / 2][2 * (x % 2) + 1];
        else return raw[2 * (x % WORDS) + 1][x / WORDS];
    }
    // LDS byte offset of the write that pair x completes, from wbase
    static constexpr uint32_t write_offset(int x) { return KC ? (x / 2) * (NT / 8) * 64 : (x / WORDS) * Q * 64; }
};

// What is done beside the MFMAs of a slice, one entry per instruction: pairs of the next slice taken apart, the planes' words written
// to LDS, the requests of the slice that takes the freed registers.
enum Kind { CVT1, LARGEST, LOW1, SUB1A, HIGH1, SUB1B, CVT2, LOW2, SUB2A, HIGH2, SUB2B, CVT3, WRITE, LOAD };
struct Op {
    int kind, operand, x, i;    // x: pair (WRITE: the pair that completes it; LOAD: the load), i: plane of a WRITE
};
template <int CAP>
struct OpList {
    Op op[CAP];
    int n;
};
template <typename OpA, typename OpB, int CAP>
constexpr OpList<CAP> list_ops()
{
    OpList<CAP> l{};
    for (int o = 0; o < 2; ++o) {
        const int pairs = o ? OpB::PAIRS : OpA::PAIRS, words = o ? OpB::WORDS : OpA::WORDS, loads = o ? OpB::NV : OpA::NV;
        const bool kc = o ? OpB::K_CONTIGUOUS : OpA::K_CONTIGUOUS;
        for (int x = 0; x < pairs; ++x) {
            for (int kind = CVT1; kind <= CVT3; ++kind) l.op[l.n++] = Op{kind, o, x, 0};
            if (x % words == words - 1)
                for (int pl = 0; pl < 3; ++pl) l.op[l.n++] = Op{WRITE, o, x, pl};
            if (kc && x % 2 == 1) l.op[l.n++] = Op{LOAD, o, x / 2, 0};
        }
        if (!kc)
            for (int v = 0; v < loads; ++v) l.op[l.n++] = Op{LOAD, o, v, 0};
    }
    return l;
}

// What each group of twelve MFMAs has to do besides: fragment reads and entries of the list of ops, N in all, the same number of
// instructions in every group.
template <int MB, int NB, int N>
struct Shares {
    // Fragments of B: where a row of blocks is long enough (four), the next slice's are read over the ones just used, a pair behind
    // the pair's MFMAs; else into registers of their own during the carried row of blocks.
    static constexpr int FB = NB > 2 ? 1 : 2, NP = NB / 2, GROUPS = MB * NP;
    static constexpr int a_reads(int g) { return g % NP == 0 && g / NP < MB ? 3 : 0; }
    static constexpr int b_reads(int g) { return FB == 1 ? (g > 0 && g <= NP ? 6 : 0) : (g < NP ? 6 : 0); }
    static constexpr int ops_before(int g)
    {
        int reads = 0, n = 0;
        for (int q = 0; q < g; ++q) {
            reads += a_reads(q) + b_reads(q);
            const int here = (N + 3 * (MB + NB)) * (q + 1) / GROUPS - reads;
            n = here > n ? here : n;
        }
        return g >= GROUPS || n > N ? N : n;
    }
};

}  // namespace planes

// A work-group: KG groups of WM x WN wavefronts; the groups take every KG-th slice each and are added at the end.
template <bool TA, bool TB, int BM, int BN, int WM, int WN, int KG>
struct PlanesCfg {
    static constexpr int GROUP = WM * WN * 64, NT = GROUP * KG;
    using A = planes::Operand<TA, BM, GROUP>;
    using B = planes::Operand<!TB, BN, GROUP>;
    static constexpr int BUF = 3 * (A::PLANE + B::PLANE);
    static constexpr int LDS_BYTES = 2 * BUF * KG;
};

template <bool TA, bool TB, int BM, int BN, int WM, int WN, int KG>
__global__ void __launch_bounds__(WM * WN * KG * 64, WM * WN * KG / 4)
gemm_planes_kernel(const GemmArgs args)
{
    using namespace planes;
    using Cfg = PlanesCfg<TA, TB, BM, BN, WM, WN, KG>;
    using OpA = typename Cfg::A;
    using OpB = typename Cfg::B;
    // a wavefront's rows: all four members of its row quads, or (tiles of 64 rows, WM = 2) two of the four members of every quad
    constexpr int MB = BM / WM / 16, NB = BN / WN / 16;  // 16 x 16 blocks of a wavefront along m and n
    constexpr int JW = BM / WM >= 64 ? 4 : 2, QW = MB / JW;
    static_assert(JW == 4 || (BM == 64 && WM == 2), "row quads, or halves of them");
    constexpr int U = 2;                                 // slices per turn of the loop: registers and LDS halves are then named at compile time
    static_assert(KG >= 1 && KG <= 3, "one to three groups of wavefronts");
    constexpr int NP = NB / 2, GROUPS = MB * NP;         // pairs of blocks, twelve MFMAs each, per slice
    constexpr int CAP = 16 * (OpA::PAIRS + OpB::PAIRS);
    constexpr OpList<CAP> ops = list_ops<OpA, OpB, CAP>();
    using Share = Shares<MB, NB, ops.n>;
    constexpr int FB = Share::FB;

    extern __shared__ __attribute__((aligned(16))) char lds[];

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave_of_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t kg = KG == 1 ? 0 : wave_of_all / (WM * WN), wave = wave_of_all % (WM * WN), tid = wave * 64 + lane;   // of the group
    const uint32_t wm = wave % WM, wn = wave / WM;
    const uint32_t l16 = lane & 15, l4 = lane >> 4;

    uint32_t wg0, wg1, tile_id, zb, nxcd;
    work_of_block(args, blockIdx.x, blockIdx.z, tile_id, zb, nxcd);
    wg_remap(tile_id, args.nwg0, args.nwg1, args.wgm, nxcd, wg0, wg1);
    const uint32_t split = zb / args.batch, batch = zb % args.batch;
    const uint32_t row0 = wg0 * BM, col0 = wg1 * BN;
    const int rows_a = (int)min((uint32_t)BM, args.m - row0), rows_b = (int)min((uint32_t)BN, args.n - col0);
    const uint32_t k_begin = split * args.k_per_split, k_end = min(args.k, k_begin + args.k_per_split);
    const int k_len = (int)(k_end - k_begin);
    const int left = k_len % BK, all = k_len / BK + (left ? 1 : 0);      // slices
    // this group's: kg, kg + KG, ..; all groups walk as many (the last may not exist: zeros)
    const int ns = (all + KG - 1) / KG;
    const bool has_partial = left && (all - 1) % KG == (int)kg;

    const uint32_t lda = args.lda, ldb = args.ldb;
    const int64_t one_a = (TA ? (int64_t)BK : (int64_t)BK * lda) * 4, one_b = (TB ? (int64_t)BK * ldb : (int64_t)BK) * 4;
    const char *gA = static_cast<const char *>(args.A) +
                     ((int64_t)batch * args.strideA + (TA ? (int64_t)row0 * lda + k_begin - 4 : (int64_t)k_begin * lda + row0 - OpA::lead(rows_a))) * 4 + kg * one_a;
    const char *gB = static_cast<const char *>(args.B) +
                     ((int64_t)batch * args.strideB + (TB ? (int64_t)k_begin * ldb + col0 - OpB::lead(rows_b) : (int64_t)col0 * ldb + k_begin - 4)) * 4 + kg * one_b;
    const int64_t stepA = one_a * KG, stepB = one_b * KG;

    OpA opA;
    OpB opB;
    opA.init(tid, lda, rows_a);
    opB.init(tid, ldb, rows_b);
    const uint32_t group_lds = kg * 2 * Cfg::BUF;
    opA.wbase += group_lds;
    opB.wbase += group_lds + 3 * OpA::PLANE;

    u32x4 rawA[OpA::NV], rawB[OpB::NV];                  // the slice that is taken apart next
    float maxA = 0.0f, maxB = 0.0f;                      // largest element seen

    // One entry of `ops`.
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    uint32_t e0 = 0, e1 = 0, p = 0, h = 0;
    uint32_t word[3][4];                                 // the planes' words of the write being put together
    auto cvt = [](uint32_t a, uint32_t b) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)}, bf16x2));
    };
    auto sub = [](uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, a) - __builtin_bit_cast(float, b)); };
    auto act = [&](auto OPERAND, auto KIND, auto X, auto I, auto &op, auto &raw, float &largest, uint32_t buf, const char *origin, int bytes) {
        using Oper = typename decltype(OPERAND)::type;
        constexpr int kind = decltype(KIND)::value, x = decltype(X)::value, w = x % Oper::WORDS;
        if constexpr (kind == CVT1) {
            e0 = Oper::first_of(raw, x);
            e1 = Oper::second_of(raw, x);
            p = word[0][w] = cvt(e0, e1);
        } else if constexpr (kind == LARGEST) {
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(largest) : "v"(e0), "v"(e1));
        } else if constexpr (kind == LOW1 || kind == LOW2) {
            h = p << 16;
        } else if constexpr (kind == HIGH1 || kind == HIGH2) {
            h = p & 0xffff0000u;
        } else if constexpr (kind == SUB1A || kind == SUB2A) {
            e0 = sub(e0, h);
        } else if constexpr (kind == SUB1B || kind == SUB2B) {
            e1 = sub(e1, h);
        } else if constexpr (kind == CVT2) {
            p = word[1][w] = cvt(e0, e1);
        } else if constexpr (kind == CVT3) {
            word[2][w] = cvt(e0, e1);
        } else if constexpr (kind == WRITE) {
            constexpr int pl = decltype(I)::value;
            char *to = lds + buf + op.wbase + Oper::write_offset(x) + pl * Oper::PLANE;
            if constexpr (Oper::WORDS == 4) *reinterpret_cast<u32x4 *>(to) = u32x4{word[pl][0], word[pl][1], word[pl][2], word[pl][3]};
            else if constexpr (Oper::WORDS == 2) *reinterpret_cast<u32x2 *>(to) = u32x2{word[pl][0], word[pl][1]};
            else *reinterpret_cast<uint32_t *>(to) = word[pl][0];
        } else if constexpr (kind == LOAD) {
            raw[x] = Oper::load(origin, op.voff[x], bytes);
        }
    };
    // entry U on the given registers; the planes go to LDS half `buf`, the requests are those of the slice at oa, ob
    auto act_on = [&](auto U, u32x4 (&ra)[OpA::NV], u32x4 (&rb)[OpB::NV], uint32_t buf, const char *oa, const char *ob, int bytes) {
        constexpr Op o = ops.op[decltype(U)::value];
        if constexpr (o.operand == 0)
            act(std::common_type<OpA>{}, std::integral_constant<int, o.kind>{}, std::integral_constant<int, o.x>{}, std::integral_constant<int, o.i>{}, opA, ra, maxA, buf, oa, bytes);
        else
            act(std::common_type<OpB>{}, std::integral_constant<int, o.kind>{}, std::integral_constant<int, o.x>{}, std::integral_constant<int, o.i>{}, opB, rb, maxB, buf, ob, bytes);
    };

    // all requests of slice x (behind the last slice: none)
    auto bytes_of = [&](int x) { return x * KG + (int)kg < all ? 0x7fffffff : 0; };
    auto load_slice = [&](u32x4 (&ra)[OpA::NV], u32x4 (&rb)[OpB::NV], int x) {
#pragma unroll
        for (int v = 0; v < OpA::NV; ++v) ra[v] = OpA::load(gA + (int64_t)x * stepA, opA.voff[v], bytes_of(x));
#pragma unroll
        for (int v = 0; v < OpB::NV; ++v) rb[v] = OpB::load(gB + (int64_t)x * stepB, opB.voff[v], bytes_of(x));
    };
    // (the partial slice is the last one there is: its requests are the last ones made)
    auto aim_at = [&](int x) {
        if (x == ns - 1 && has_partial) {
            opA.aim_partial(lda, left);
            opB.aim_partial(ldb, left);
        }
    };
    auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // fragments
    const uint32_t frag_lane = l16 * 64 + ((l4 ^ swizzle(l16)) << 4);
    const uint32_t fragA = group_lds + frag_lane + (JW == 4 ? wm * QW : 2 * wm) * 1024, fragB = group_lds + frag_lane + 3 * OpA::PLANE + wn * NB * 1024;
    // a wavefront's block mb along m: quads' member j = mb / QW (plus 2 wm where JW = 2), 16 quads from block mb % QW on
    auto block_a = [](int mb) { return (mb / QW) * (BM / 64) + mb % QW; };
    u32x4 fa[2][3], fb[FB][NB][3];
    f32x4 big[MB][NB], small[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) big[i][j] = small[i][j] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
        fa[1][pl] = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < NB; ++j) fb[0][j][pl] = fb[FB - 1][j][pl] = u32x4{0, 0, 0, 0};
    }
    auto read_a = [&](u32x4 &f, int mb, int pl, uint32_t buf) {
        f = *reinterpret_cast<const u32x4 *>(lds + buf + fragA + block_a(mb) * 1024 + pl * OpA::PLANE);
    };
    auto read_b = [&](u32x4 &f, int nb, int pl, uint32_t buf) {
        f = *reinterpret_cast<const u32x4 *>(lds + buf + fragB + nb * 1024 + pl * OpB::PLANE);
    };
    auto mfma = [](const u32x4 &n_side, const u32x4 &m_side, f32x4 &c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, n_side), __builtin_bit_cast(bf16x8, m_side), c, 0, 0, 0);
    };

    const char *ahead_a = gA + 2 * stepA, *ahead_b = gB + 2 * stepB;     // of the slice requested next
    // One slice.  Its phase PH says which registers and which half of LDS hold what; phases count so that the last slice has phase 0.
    auto slice = [&](auto PH, auto LAST, int s) {
        constexpr int ph = decltype(PH)::value, par = ph & 1;
        constexpr bool last = decltype(LAST)::value;
        constexpr uint32_t here = par ? Cfg::BUF : 0, next = par ? 0 : Cfg::BUF;
        if constexpr (!last) {
            if (s + 2 == ns && has_partial) {
                opA.fix_partial(rawA, left);
                opB.fix_partial(rawB, left);
            }
            aim_at(s + 2);
        }
        const int bytes = bytes_of(s + 2);
        // A group: two neighbouring blocks, six MFMAs each, with its share of what else there is to do spread over
        // them: first the fragment reads that the next groups need, then entries of `ops`.
        static_for<GROUPS + (last ? NP : 0)>([&](auto G) {
            constexpr int g = decltype(G)::value, turn = g / NP, h = g % NP;
            constexpr int mb = turn == 0 ? MB - 1 : turn - 1;             // turn 0: the last row of blocks of the slice before
            constexpr int a_reads = Share::a_reads(g), reads = a_reads + Share::b_reads(g);
            constexpr int from = last ? 0 : Share::ops_before(g), to = last ? 0 : Share::ops_before(g + 1), acts = reads + to - from;
            static_for<12>([&](auto I) {
                // block by block, each MFMA with one operand of the one before it, the small products in a chain: a power-limited chip
                // runs this order fastest (NT 4096^3 546 -> 526 us against alternating between the two blocks)
                constexpr int i = decltype(I)::value, nb = 2 * h + i / 6;
                const u32x4(&a)[3] = fa[mb & 1];
                const u32x4(&b)[3] = fb[FB == 1 ? 0 : turn == 0 ? par ^ 1 : par][nb];
                if constexpr (i % 6 == 0) mfma(b[2], a[0], small[mb][nb]);
                if constexpr (i % 6 == 1) mfma(b[1], a[0], small[mb][nb]);
                if constexpr (i % 6 == 2) mfma(b[1], a[1], small[mb][nb]);
                if constexpr (i % 6 == 3) mfma(b[0], a[1], small[mb][nb]);
                if constexpr (i % 6 == 4) mfma(b[0], a[2], small[mb][nb]);
                if constexpr (i % 6 == 5) mfma(b[0], a[0], big[mb][nb]);
                constexpr int at = i * acts / 12, end = (i + 1) * acts / 12;
                static_for<end - at>([&](auto D) {
                    constexpr int d = at + decltype(D)::value;
                    if constexpr (d < a_reads) {
                        read_a(fa[turn & 1][d], turn, d, here);
                    } else if constexpr (d < reads) {
                        constexpr int e = d - a_reads, nbr = (FB == 1 ? 2 * (g - 1) : 2 * h) + e % 2;
                        read_b(fb[FB == 1 ? 0 : par][nbr][e / 2], nbr, e / 2, here);
                    } else {
                        act_on(std::integral_constant<int, from + d - reads>{}, rawA, rawB, next, ahead_a, ahead_b, bytes);
                    }
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        ahead_a += stepA;
        ahead_b += stepB;
        barrier();
    };

    // slice 0, of phase `first`, is taken apart ahead of the loop
    const int first = (U - (ns - 1) % U) % U;
    static_for<U>([&](auto PH) {
        constexpr int ph = decltype(PH)::value;
        constexpr uint32_t here = ph & 1 ? Cfg::BUF : 0;
        if (first != ph) return;
        aim_at(0);
        load_slice(rawA, rawB, 0);
        if (ns == 1 && has_partial) {
            opA.fix_partial(rawA, left);
            opB.fix_partial(rawB, left);
        }
        aim_at(1);
        static_for<ops.n>([&](auto U) {
            act_on(U, rawA, rawB, here, gA + stepA, gB + stepB, bytes_of(1));
        });
    });
    barrier();

    for (int at = -first; at < ns - 1; at += U) {
        asm volatile("" : "+s"(at));                      // (the first turn is not to be taken out of the loop)
        static_for<U>([&](auto PH) {
            constexpr int ph = decltype(PH)::value;
            if (ph == U - 1 || at + ph >= 0) slice(PH, std::false_type{}, at + ph);
        });
    }
    slice(std::integral_constant<int, 0>{}, std::true_type{}, ns - 1);

    // ---- C --------------------------------------------------------------------------------------------------------
    // A lane has columns 4 * l4 + i of each block of 16 (physical) and row quads l16 of each block of quads.
    // Row (of the tile) of member j of quad q, as it was loaded: KC operands repeat their last row past the edge, the others' quads are moved up.
    auto row_a = [&](int q, int j) { return TA ? min(4 * q + j, rows_a - 1) : OpA::quad_row(q, rows_a) + j; };
    auto row_b = [&](int q, int j) { return !TB ? min(4 * q + j, rows_b - 1) : OpB::quad_row(q, rows_b) + j; };
    constexpr int QB = BN / 4;
    typedef f32x4 __attribute__((aligned(4))) f32x4_u;
    typedef f32x2 __attribute__((aligned(4))) f32x2_u;
    using Rows = typename std::conditional<JW == 4, f32x4, f32x2>::type;
    using Rows_u = typename std::conditional<JW == 4, f32x4_u, f32x2_u>::type;
    constexpr int NE = KG == 1 ? NB : NB / 2;            // columns of blocks a wavefront stores, from physical column n0 on (see below)
    const bool stores = KG < 3 || kg < 2;
    const int n0 = (int)((wn * NB + (KG < 3 || kg < 2 ? kg : 0) * NE) * 16);
    const int j0 = JW == 4 ? 0 : 2 * (int)wm;            // first member of its quads
    const bool to_ws = args.splits > 1;
    const uint32_t ldo = to_ws ? args.m : args.ldc;
    float *out = to_ws ? args.ws + ((size_t)split * args.batch + batch) * (size_t)args.m * args.n
                       : static_cast<float *>(args.C) + (int64_t)batch * args.strideC;
    const float alpha = to_ws ? 1.0f : args.alpha, beta = to_ws ? 0.0f : args.beta;
    auto quad = [&](int qi) { return (int)((JW == 4 ? wm * QW : 0) + qi) * 16 + (int)l16; };
    auto column = [&](int nb, int i) { return row_b((n0 + nb * 16) % QB + 4 * (int)l4 + i, (n0 + nb * 16) / QB); };
    auto column_in = [&](int nb, int i) {
        const int q = (n0 + nb * 16) % QB + 4 * (int)l4 + i, j = (n0 + nb * 16) / QB;
        return stores && 4 * q < rows_b && (TB ? column(nb, i) >= 4 * q : 4 * q + j < rows_b);
    };
    auto c_at = [&](int nb, int i, int qi) { return out + (size_t)(col0 + column(nb, i)) * ldo + row0 + 4 * quad(qi) + j0; };
    // a quad that the edge cuts: member j holds row quad_row + j (memory contiguous along m) or row 4 q + j, `up` of them further up
    auto up = [&](int q) { return TA ? 0 : 4 * q - OpA::quad_row(q, rows_a); };
    auto member_in = [&](int q, int j) { return j0 + j >= up(q) && 4 * q + j0 + j - up(q) < rows_a; };
    // the old C, all of it requested before anything else is done (one round trip to memory; a block of columns at a time, four; the
    // elements of cut quads, where they are used, were a round trip each: NT 1639 x 1845 x 256 with beta 21.6 -> 17.2 us)
    Rows old[NE][4][QW];
    if (beta != 0.0f) {                                  // beta == 0: C is never read
#pragma unroll
        for (int nb = 0; nb < NE; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int qi = 0; qi < QW; ++qi)
                    if (column_in(nb, i) && 4 * quad(qi) + 4 <= rows_a) old[nb][i][qi] = *reinterpret_cast<const Rows_u *>(c_at(nb, i, qi));
        if (rows_a % 4 != 0) {
#pragma unroll
            for (int nb = 0; nb < NE; ++nb)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int qi = 0; qi < QW; ++qi) {
                        const int q = quad(qi);
                        const float *p = c_at(nb, i, qi) - up(q);
                        if (column_in(nb, i) && 4 * q < rows_a && 4 * q + 4 > rows_a)
#pragma unroll
                            for (int j = 0; j < JW; ++j)
                                if (member_in(q, j)) old[nb][i][qi][j] = p[j];
                    }
        }
    }

    // ---- the sums ---------------------------------------------------------------------------------------------------
    // Two groups: each wavefront hands half of its columns of blocks to the wavefront of the same rows and columns in the other group and
    // adds what it gets to the rest (the first group's sum first).  A third group hands one half to each of them, which add it behind their
    // own, and goes on with zeros that it does not store.  From here on a wavefront has NE columns of blocks, from n0 on.
    f32x4 sum[MB][NE];
    if constexpr (KG == 1) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NE; ++j) sum[i][j] = big[i][j] + small[i][j];
    } else {
        // (the last slice's barrier is behind its last read)  half h of what group g hands on:
        auto half = [&](uint32_t g, uint32_t h) {
            return reinterpret_cast<f32x4 *>(lds) + ((g < 2 ? g : 2 + h) * WM * WN + wave) * (MB * NE * 64) + lane;
        };
        static_for<KG>([&](auto K) {
            constexpr int k = decltype(K)::value;
            if ((int)kg != k) return;
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NE; ++j) {
                    if constexpr (k == 2) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) half(2, h)[(i * NE + j) * 64] = big[i][h * NE + j] + small[i][h * NE + j];
                        sum[i][j] = f32x4{0, 0, 0, 0};
                    } else {
                        half(k, 0)[(i * NE + j) * 64] = big[i][(k ^ 1) * NE + j] + small[i][(k ^ 1) * NE + j];
                        sum[i][j] = big[i][k * NE + j] + small[i][k * NE + j];
                    }
                }
        });
        barrier();
        if (stores) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NE; ++j) {
                    sum[i][j] += half(kg ^ 1, 0)[(i * NE + j) * 64];
                    if constexpr (KG == 3) sum[i][j] += half(2, kg)[(i * NE + j) * 64];
                }
        }
        barrier();
    }

    // ---- what the planes cannot hold -----------------------------------------------------------------------------
    // (a) An infinity, a NaN or an element that rounds to a bf16 infinity leaves no finite accumulator in its row or column of the tile
    //     (inf - inf and inf * 0 are NaN), and so does a sum that overflows.
    // (b) bf16 is granular to 2^-133: planes of elements below 2^-109 lose bits, and elements below 2^-134 vanish.  Of a sum that is, at
    //     most, k * 2^-133 * the largest element of the tile's operands, so only a sum that is not 2^25 times that may show it, an exact zero
    //     among them.  Ordinary data has such sums too -- rows of zeros, of zeros and small integers, at k = 4096 anything below 2^-126 where no
    //     element reaches 2^-30, 2^-76 where none reaches 2^20, 2^-36 up to 2^60 --, so then the work-group looks through its rows and columns
    //     for elements below 2^-109: one more pass over the operands, bound by what a CU pulls from the L2 (a row of zeros in every tile, us
    //     without it / with it: NN 1024^3 21.8 / 26.6, 2048^3 92 / 113, 4096^3 556 / 649, TN 640 x 384 x 10000 40.5 / 64).
    // (c) A sum below k * 2^-138 is within reach of fp32's own smallest numbers, where the small products end.
    // With (a), (c), or an element that (b) finds, the work-group computes its tile again with fp32 MFMAs.
    float poison = 0.0f;
    uint32_t least = 0xffffffffu, most = 0;               // of 2 |sum| - 1 as bits: zeros last
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NE; ++j) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = sum[i][j][e];             // (the bits of sum[i][j][e] would be those of element 0: __builtin_bit_cast takes the whole vector)
                poison = __builtin_fmaf(x, 0.0f, poison);
                const uint32_t bits = (__builtin_bit_cast(uint32_t, x) << 1) - 1;
                least = min(least, bits);
                most = max(most, bits);
            }
        }
    const float k_f = (float)k_len;
    auto below = [&](float limit) { return least < __builtin_bit_cast(uint32_t, limit) << 1; };
    auto any = [](bool x) { return __builtin_amdgcn_ballot_w64(x) != 0; };
    const float largest = fmaxf(maxA, maxB);
    uint32_t flags = any(!(poison == 0.0f)) || any(below(k_f * 0x1p-138f)) ? 1 : 0;
    flags |= any(below(k_f * 0x1p-88f)) ? 2 : 0;
    flags |= any(below(k_f * 0x1p-48f)) ? 4 : 0;
    flags |= any(below(k_f * 0x1p+20f)) ? 8 : 0;
    flags |= any(largest >= 0x1p-30f) ? 16 : 0;
    flags |= any(largest >= 0x1p+20f) ? 32 : 0;
    flags |= any(largest >= 0x1p+60f) ? 64 : 0;
    flags |= stores && any(most == 0xffffffffu) ? 128 : 0;
    flags |= any(maxA != 0.0f) ? 256 : 0;
    flags |= any(maxB != 0.0f) ? 512 : 0;
    uint32_t *shared_flags = reinterpret_cast<uint32_t *>(lds);
    auto of_all = [&](uint32_t x) {                       // x of all wavefronts, or-ed
        if (lane == 0) shared_flags[wave_of_all] = x;
        barrier();
        x = 0;
#pragma unroll
        for (int w = 0; w < WM * WN * KG; ++w) x |= shared_flags[w];
        shared_flags += WM * WN * KG;
        return (uint32_t)__builtin_amdgcn_readfirstlane(x);
    };
    flags = of_all(flags);
    // (bits 1-3: a sum below the limit; bits 4-6: an element that the limit holds for)
    bool again = flags & 1;
    if (!again && ((flags >> 4 & flags >> 1 & 7) || (flags & (128 | 256 | 512)) == (128 | 256 | 512))) {
        // the requests of the loop once more (their offsets anew: kept, they would cost the loop registers)
        uint32_t t = tid;
        asm volatile("" : "+v"(t));
        opA.init(t, lda, rows_a);
        opB.init(t, ldb, rows_b);
        uint32_t smallest = 0xffffffffu;                  // of 2 |element| - 1 as bits
        auto look = [&](int x) {
            load_slice(rawA, rawB, x);
#pragma unroll
            for (int v = 0; v < OpA::NV; ++v)
#pragma unroll
                for (int e = 0; e < 4; ++e) smallest = min(smallest, (rawA[v][e] << 1) - 1);
#pragma unroll
            for (int v = 0; v < OpB::NV; ++v)
#pragma unroll
                for (int e = 0; e < 4; ++e) smallest = min(smallest, (rawB[v][e] << 1) - 1);
        };
#pragma unroll 4
        for (int x = 0; x < ns - 1; ++x) look(x);
        aim_at(ns - 1);
        look(ns - 1);
        again = of_all(any(smallest < __builtin_bit_cast(uint32_t, 0x1p-109f) << 1));
    }

    // Steps of 16 k, four to a lane (in one load where the operand is contiguous along k), straight to registers and DEPTH steps ahead of their MFMAs.
    // Runs of 128 k, so that no sum is less exact than those of the kernels that planes replace, whose runs are as long or longer.
    // The time is that of the planes and then the fp32 MFMAs' own.  us, ordinary data / a NaN in every tile (there, element by element and four k
    // at a time: in brackets) / the fp32 MFMA kernels: NN 4096^3 556 / 1479 (3110) / 927, TN 567 / 1502 (4012) / 914, NT with alpha and beta 635 / 1598
    // (2610) / 941, NN 2048^3 92 / 235 (526) / 136, NN 1024^3 21.8 / 51.6 (184) / 25.2, TN 640 x 384 x 10000 40.5 / 130 (379) / 54.  (One run of all k: 5 %
    // less at 4096^3.)
    if (again && stores) {
        constexpr int DEPTH = MB * NE >= 16 ? 2 : 4;
        const char *a0 = gA - kg * one_a + (TA ? 16 : 0), *b0 = gB - kg * one_b + (TB ? 0 : 16);
        // byte offsets of a lane's first k (A contiguous along the rows: of the JW rows that it has of a quad, for the blocks of all of them)
        constexpr int LA = TA ? MB : QW;
        f32x4 total[MB][NE];                              // of whole runs
        uint32_t at_a[LA], at_b[NE];
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const uint32_t r = row_a(quad(i % QW), j0 + i / QW) + OpA::lead(rows_a);
            at_a[i] = (TA ? r * lda + 4 * l4 : 4 * l4 * lda + r) * 4;
        }
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            const int p = n0 + j * 16 + l16;
            const uint32_t r = row_b(p % QB, p / QB) + OpB::lead(rows_b);
            at_b[j] = (TB ? 4 * l4 * ldb + r : r * ldb + 4 * l4) * 4;
#pragma unroll
            for (int i = 0; i < MB; ++i) sum[i][j] = total[i][j] = f32x4{0, 0, 0, 0};
        }
        const int steps = k_len / 16, rest = k_len % 16;
        const int64_t step_a = (TA ? (int64_t)16 : (int64_t)16 * lda) * 4, step_b = (TB ? (int64_t)16 * ldb : (int64_t)16) * 4;
        struct Step {
            float a[MB][4], b[NE][4];
        } x[DEPTH];
        // N elements in a row
        auto load = [](auto N, auto &&put, const char *origin, uint32_t off, uint32_t more) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(origin), 0, 0x7fffffff, 0x00020000);
            auto number = [](uint32_t w) { return __builtin_bit_cast(float, w); };
            if constexpr (decltype(N)::value == 4) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, more, 0);
                static_for<4>([&](auto E) { put(E) = number(v[decltype(E)::value]); });
            } else if constexpr (decltype(N)::value == 2) {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, more, 0);
                static_for<2>([&](auto E) { put(E) = number(v[decltype(E)::value]); });
            } else {
                put(std::integral_constant<int, 0>{}) = number(__builtin_amdgcn_raw_buffer_load_b32(r, off, more, 0));
            }
        };
        constexpr std::integral_constant<int, 1> one;
        constexpr std::integral_constant<int, 4> four;
        constexpr std::integral_constant<int, JW> rows;
        auto fetch = [&](Step &to, int s) {
            const char *oa = a0 + s * step_a, *ob = b0 + s * step_b;
            static_for<LA>([&](auto I) {
                constexpr int i = decltype(I)::value;
                if constexpr (TA) load(four, [&](auto T) -> float & { return to.a[i][decltype(T)::value]; }, oa, at_a[i], 0);
                else static_for<4>([&](auto T) {
                    load(rows, [&](auto J) -> float & { return to.a[decltype(J)::value * QW + i][decltype(T)::value]; }, oa, at_a[i], decltype(T)::value * lda * 4);
                });
            });
            static_for<NE>([&](auto J) {
                constexpr int j = decltype(J)::value;
                if constexpr (!TB) load(four, [&](auto T) -> float & { return to.b[j][decltype(T)::value]; }, ob, at_b[j], 0);
                else static_for<4>([&](auto T) { load(one, [&](auto) -> float & { return to.b[j][decltype(T)::value]; }, ob, at_b[j], decltype(T)::value * ldb * 4); });
            });
        };
        auto multiply = [&](const Step &of) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NE; ++j) sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(of.b[j][t], of.a[i][t], sum[i][j], 0, 0, 0);
        };
        if (steps >= DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) fetch(x[d], d);
        }
        auto end_run = [&] {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NE; ++j) {
                    total[i][j] += sum[i][j];
                    sum[i][j] = f32x4{0, 0, 0, 0};
                }
        };
        int s = 0;
        for (; s + DEPTH <= steps; s += DEPTH) {
            static_for<DEPTH>([&](auto D) {
                constexpr int d = decltype(D)::value;
                multiply(x[d]);
                fetch(x[d], min(s + d + DEPTH, steps - 1));
            });
            if ((s + DEPTH) % 8 == 0) end_run();
        }
        for (; s < steps; ++s) {
            fetch(x[0], s);
            multiply(x[0]);
        }
        if (rest > 0) {
            // element by element; an offset outside the buffer brings zero
            const char *oa = a0 + steps * step_a, *ob = b0 + steps * step_b;
            static_for<4>([&](auto T) {
                constexpr int t = decltype(T)::value;
                const bool in = (int)(4 * l4) + t < rest;
                static_for<MB>([&](auto I) {
                    constexpr int i = decltype(I)::value;
                    load(one, [&](auto) -> float & { return x[0].a[i][t]; }, oa, in ? at_a[TA ? i : i % QW] + (TA ? 0 : i / QW * 4) : 0x80000000u, (TA ? t : t * lda) * 4);
                });
                static_for<NE>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    load(one, [&](auto) -> float & { return x[0].b[j][t]; }, ob, in ? at_b[j] : 0x80000000u, (TB ? t * ldb : t) * 4);
                });
            });
            multiply(x[0]);
        }
        end_run();
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NE; ++j) sum[i][j] = total[i][j];
    }

    // ---- and out ----------------------------------------------------------------------------------------------------
#pragma unroll
    for (int nb = 0; nb < NE; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!column_in(nb, i)) continue;
#pragma unroll
            for (int qi = 0; qi < QW; ++qi) {
                const int q = quad(qi);
                float *at = c_at(nb, i, qi);
                Rows v;
#pragma unroll
                for (int j = 0; j < JW; ++j) {
                    v[j] = alpha * sum[j * QW + qi][nb][i];
                    if (beta != 0.0f) v[j] = __builtin_fmaf(beta, old[nb][i][qi][j], v[j]);
                }
                if (4 * q + 4 <= rows_a) {
                    *reinterpret_cast<Rows_u *>(at) = v;
                } else if (4 * q < rows_a) {
                    float *p = at - up(q);
#pragma unroll
                    for (int j = 0; j < JW; ++j)
                        if (member_in(q, j)) p[j] = v[j];
                }
            }
        }
}

}  // namespace mmbo
