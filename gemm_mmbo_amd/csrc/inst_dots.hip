// Instantiates the fp64 kernel for small results of long sums for one tile row: compile with -DMMBO_TILE=<row>
#include <atomic>

#include "configs.hpp"
#include "gemm_dots.hpp"
#include "launch.hpp"

#ifndef MMBO_TILE
#error "MMBO_TILE selects what this translation unit instantiates"
#endif

namespace mmbo {

namespace {
constexpr DotsRow R = kDotsTiles[MMBO_TILE];
static_assert(dots::kStep == kDotsStep, "");

template <bool TA, bool TB>
hipError_t launch_one(const GemmArgs &args, hipStream_t stream)
{
    using Cfg = DotsCfg<R.fm, R.fn, kDotsWaves, R.depth>;
    auto kernel = gemm_dots_kernel<TA, TB, R.fm, R.fn, kDotsWaves, R.depth>;
    static_assert(Cfg::LDS_BYTES <= 160 * 1024, "the rings do not fit the 160 KB of LDS");
    static std::atomic<bool> attr_set[64];           // zero-initialised; several host threads may race to set it: harmless
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64 && !attr_set[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set[dev].store(true, std::memory_order_release);
    }
    return launch_kernel(kernel, dim3(args.batch, args.nwg0 * args.nwg1, 1), dim3(kDotsWaves * 64), Cfg::LDS_BYTES, stream, args);
}
}  // namespace

template <>
hipError_t launch_dots<MMBO_TILE>(int transA, int transB, const GemmArgs &args, hipStream_t stream)
{
    if (!transA && !transB) return launch_one<false, false>(args, stream);
    if (!transA && transB) return launch_one<false, true>(args, stream);
    if (transA && !transB) return launch_one<true, false>(args, stream);
    return launch_one<true, true>(args, stream);
}

}  // namespace mmbo
