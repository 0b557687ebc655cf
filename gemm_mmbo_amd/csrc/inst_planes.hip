// Instantiates the kernel on three bf16 planes (fp32 operands) for one tile row: compile with -DMMBO_TILE=<row>
#include <atomic>

#include "configs.hpp"
#include "gemm_planes.hpp"
#include "launch.hpp"

#ifndef MMBO_TILE
#error "MMBO_TILE selects what this translation unit instantiates"
#endif

namespace mmbo {

namespace {
constexpr PlanesRow R = kPlanesTiles[MMBO_TILE];

template <bool TA, bool TB>
hipError_t launch_one(const GemmArgs &args, hipStream_t stream)
{
    using Cfg = PlanesCfg<TA, TB, R.bm, R.bn, R.wm, R.wn, R.kg>;
    auto kernel = gemm_planes_kernel<TA, TB, R.bm, R.bn, R.wm, R.wn, R.kg>;
    static_assert(Cfg::LDS_BYTES <= 160 * 1024, "two slices of planes do not fit the 160 KB of LDS");
    static std::atomic<bool> attr_set[64];           // zero-initialised; several host threads may race to set it: harmless
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64 && !attr_set[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
        if (e != hipSuccess) return e;
        attr_set[dev].store(true, std::memory_order_release);
    }
    dim3 grid(args.nwg0 * args.nwg1, 1, args.batch * args.splits);
    return launch_kernel(kernel, grid, dim3(Cfg::NT), Cfg::LDS_BYTES, stream, args);
}
}  // namespace

template <>
hipError_t launch_planes<MMBO_TILE>(int transA, int transB, const GemmArgs &args, hipStream_t stream)
{
    if (!transA && !transB) return launch_one<false, false>(args, stream);
    if (!transA && transB) return launch_one<false, true>(args, stream);
    if (transA && !transB) return launch_one<true, false>(args, stream);
    return launch_one<true, true>(args, stream);
}

}  // namespace mmbo
