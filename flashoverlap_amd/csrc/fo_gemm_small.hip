// The 64x64 macro tile of the GEMM (kernel body: fo_gemm_body.h), for outputs of which even 128x128 tiles
// leave most of the GPU idle and whose K is too short for the split over K to pay (it costs a second
// launch and the parts' way through memory).  Smaller than every layout tile: for the plain GEMM and for
// calls that signal nothing.  Bound by the copies' latency and the L2, like the 128x128 tile, but a
// k-step moves half as much per CU.
#include "fo_gemm_body.h"

namespace fo {

template <typename T, int MODE, bool EDGE>
__global__ void __launch_bounds__(256) gemm_small_kernel(const GemmParams p) {
    gemm_body<T, 64, 64, MODE, 1, MODE == kPlain ? 0 : 1, EDGE>(p);
}

template <typename T, int MODE, bool EDGE>
static int launch_t(const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return launch_gemm_kernel<gemm_small_kernel<T, MODE, EDGE>, 5 * 64 * kRowBytes>(p, timer, stream);
}

template <typename T>
static int launch_mode(int mode, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    if (mode == kSignal) return launch_t<T, kSignal, false>(p, timer, stream);
    if (mode == kScatter) return launch_t<T, kScatter, false>(p, timer, stream);
    return edge ? launch_t<T, kPlain, true>(p, timer, stream) : launch_t<T, kPlain, false>(p, timer, stream);
}

int launch_gemm_small(int mode, int dtype, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return dtype == FO_F16 ? launch_mode<_Float16>(mode, edge, p, timer, stream) : launch_mode<__bf16>(mode, edge, p, timer, stream);
}

}  // namespace fo
