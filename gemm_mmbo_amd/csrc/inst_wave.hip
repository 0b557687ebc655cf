// Instantiates the split-by-wavefront kernel for one (element type, tile row): compile with
//   -DMMBO_DTYPE=<0|1|2> -DMMBO_TILE=<row>
#include <atomic>

#include "configs.hpp"
#include "gemm_wave.hpp"
#include "launch.hpp"

#ifndef MMBO_DTYPE
#error "MMBO_DTYPE and MMBO_TILE select what this translation unit instantiates"
#endif

namespace mmbo {

namespace {
using ElemT = typename std::conditional<MMBO_DTYPE == 0, float, typename std::conditional<MMBO_DTYPE == 1, half_t, double>::type>::type;
static_assert(MMBO_TILE < wave_tiles(MMBO_DTYPE), "a tile this type has");
constexpr WaveRow R = kWaveTiles[MMBO_TILE];
constexpr int kMaxWaves = wave_max_waves(R);

template <bool TA, bool TB>
hipError_t launch_one(const GemmArgs &args, int waves, hipStream_t stream)
{
    using Cfg = WaveCfg<ElemT, TA, TB, R.bm, R.bn, R.depth>;
    auto kernel = gemm_wave_kernel<ElemT, TA, TB, R.bm, R.bn, R.depth, kMaxWaves>;
    static_assert(Cfg::lds_bytes(kMaxWaves) <= 160 * 1024, "the rings do not fit the 160 KB of LDS");
    if (waves < 1 || waves > kMaxWaves) return hipErrorInvalidValue;
    static std::atomic<bool> attr_set[64];           // zero-initialised; several host threads may race to set it: harmless
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64 && !attr_set[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                Cfg::lds_bytes(kMaxWaves));
        if (e != hipSuccess) return e;
        attr_set[dev].store(true, std::memory_order_release);
    }
    dim3 grid(args.batch, args.nwg0 * args.nwg1, args.splits);
    return launch_kernel(kernel, grid, dim3(waves * 64), Cfg::lds_bytes(waves), stream, args);
}
}  // namespace

template <>
hipError_t launch_wave<MMBO_DTYPE, MMBO_TILE>(int transA, int transB, const GemmArgs &args, int waves, hipStream_t stream)
{
    if (!transA && !transB) return launch_one<false, false>(args, waves, stream);
    if (!transA && transB) return launch_one<false, true>(args, waves, stream);
    if (transA && !transB) return launch_one<true, false>(args, waves, stream);
    return launch_one<true, true>(args, waves, stream);
}

}  // namespace mmbo
