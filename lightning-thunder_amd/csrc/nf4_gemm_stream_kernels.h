// The launches of stream_kernel for one element type, with fp32 or nested absmax: included by one source file per pair, so
// that they compile side by side.  STREAM_F16 / STREAM_NESTED say which.
#include "nf4_gemm_stream.h"

namespace nf4 {
namespace stream {
namespace {

constexpr int MAX_DEVICES = 64;

template <bool ABS4, int BM, int WN>
hipError_t launch_one(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream) {
    using T = Shape<STREAM_NESTED, BM, WN>;
    if constexpr (!T::FITS) {
        return hipErrorInvalidValue;
    } else {
        static bool ready[MAX_DEVICES] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
        auto kern = stream_kernel<STREAM_F16, STREAM_NESTED, ABS4, BM, WN>;
        if (!ready[dev]) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM_BYTES);
            if (e != hipSuccess) return e;
            ready[dev] = true;
        }
        const int units = (a.K / STEP_K + 3) / 4, groups = p.splits * T::WK;
        uint32_t* counters = static_cast<uint32_t*>(a.workspace);
        float* partials = p.splits > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(a.workspace) + GEMV_COUNTER_REGION_BYTES) : nullptr;
        hipLaunchKernelGGL(kern, dim3((unsigned)p.n_tiles, (unsigned)p.splits, (unsigned)p.m_tiles), dim3(THREADS), T::SMEM_BYTES, stream, a,
                           p.splits, units / groups, units % groups, counters, partials);
        return hipGetLastError();
    }
}

template <bool ABS4>
hipError_t launch_any(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream) {
    switch (p.bm * 16 + p.wn) {
        case 16 * 16 + 2: return launch_one<ABS4, 16, 2>(a, p, stream);
        case 16 * 16 + 4: return launch_one<ABS4, 16, 4>(a, p, stream);
        case 16 * 16 + 8: return launch_one<ABS4, 16, 8>(a, p, stream);
        case 32 * 16 + 2: return launch_one<ABS4, 32, 2>(a, p, stream);
        case 32 * 16 + 4: return launch_one<ABS4, 32, 4>(a, p, stream);
        case 32 * 16 + 8: return launch_one<ABS4, 32, 8>(a, p, stream);
        case 64 * 16 + 4: return launch_one<ABS4, 64, 4>(a, p, stream);
        case 64 * 16 + 8: return launch_one<ABS4, 64, 8>(a, p, stream);
        case 128 * 16 + 8: return launch_one<ABS4, 128, 8>(a, p, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t STREAM_LAUNCH(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream) {
    return a.block_log2 == 6 && a.K % 256 == 0 ? launch_any<true>(a, p, stream) : launch_any<false>(a, p, stream);
}

}  // namespace stream
}  // namespace nf4
