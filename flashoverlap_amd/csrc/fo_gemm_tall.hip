// The 256x128 macro tile of the GEMM (kernel body: fo_gemm_body.h), for outputs of which 256x256 tiles
// would be too few to fill the GPU.
//
// 128x128 tiles do fill it, but move twice the operand bytes per flop from the L2 to the LDS that
// 256x256 tiles move, and the CUs then take all their L2 gives (0.46 us per k-step of 64 and tile,
// 70 bytes per ns and CU).  This tile moves half as much again as the 256x256 one; its k-step is bound
// by the LDS (96 KiB of fragment reads and 48 KiB of copies against 1024 cycles of MFMAs) and, where the
// operands come from HBM, by the copies' latency.  A B panel is half an A panel here, so three A and four B panels
// fill the 160 KiB and the copies run three panels ahead.  Plain GEMM and norm with operands that the memory-side cache
// does not hold, us, with two panels ahead / three: 1024x8192x3584 bf16 61.6 / 57.3, 2041x4096x7168 fp16 114.3 / 107.9,
// 600x4992x7360 98.9 / 81.6, 3687x1000x7600 bf16 137.7 / 103.4, 1152x4160x3008 40.7 / 41.5; with operands that it
// holds, 2048x4096x7168 96.8 / 95.5.
#include "fo_gemm_body.h"

namespace fo {

constexpr int kTallDepth = 3;
static_assert(kTurnFrom / kXcds >= kTallDepth, "the first panels, as many as the ring is deep, are copied without a turn");

template <typename T, int MODE, bool EDGE>
__global__ void __launch_bounds__(256) gemm_tall_kernel(const GemmParams p) {
    gemm_body<T, 256, 128, MODE, 1, MODE == kPlain ? 0 : 1, EDGE, kTallDepth>(p);
}

template <typename T, int MODE, bool EDGE>
static int launch_t(const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return launch_gemm_kernel<gemm_tall_kernel<T, MODE, EDGE>, ring_bytes(256, 128, kTallDepth)>(p, timer, stream);
}

template <typename T>
static int launch_mode(int mode, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    if (mode == kSignal) return launch_t<T, kSignal, false>(p, timer, stream);
    if (mode == kScatter) return launch_t<T, kScatter, false>(p, timer, stream);
    return edge ? launch_t<T, kPlain, true>(p, timer, stream) : launch_t<T, kPlain, false>(p, timer, stream);
}

int launch_gemm_tall(int mode, int dtype, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return dtype == FO_F16 ? launch_mode<_Float16>(mode, edge, p, timer, stream) : launch_mode<__bf16>(mode, edge, p, timer, stream);
}

}  // namespace fo
