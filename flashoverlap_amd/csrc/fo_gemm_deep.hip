// The GEMM with a deeper ring (kernel body: fo_gemm_body.h): four panels ahead of the one being multiplied
// instead of two.  For the 64x64 macro tile, and for the 128x128 one where no CU gets a second workgroup.
//
// 64x64 is for outputs of which even 128x128 tiles leave most of the GPU idle and whose K is too short for
// the split over K to pay (it costs a second launch and the parts' way through memory).  It is smaller than
// every layout tile: for the plain GEMM and for calls that signal nothing.
//
// Both are bound by the latency of the copies: a k-step of a 128x128 tile is a quarter of a microsecond of
// MFMAs and a copy from HBM takes one to two.  Two panels ahead of every CU are 8 MiB of the weights in
// flight, or 4 TB/s; four panels, 144 KiB of LDS at 128x128 and 72 (two workgroups to a CU) at 64x64, are twice
// that.  Kernel alone, two -> four panels, bf16: 1024x1024x1024 (64x64) 8.9 -> 6.1 us, 85x7680x7616 in 4 parts
// 31.9 -> 25.6, 128x4096x7168 in 8 16.3 -> 14.5 (4 TB/s), 256x4096x7168 in 4 25.3 -> 22.5; whole plain calls:
// 1664x2048x3904 32.0 -> 26.7, 397x3512x1408 11.6 -> 10.6.
#include "fo_gemm_body.h"

namespace fo {

constexpr int kDeep = 4;

template <typename T, int MT, int MODE, bool EDGE>
__global__ void __launch_bounds__(256) gemm_deep_kernel(const GemmParams p) {
    gemm_body<T, MT, MT, MODE, 1, MODE == kPlain ? 0 : 1, EDGE, kDeep>(p);
}

template <typename T, int MT, int MODE, bool EDGE>
static int launch_t(const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return launch_gemm_kernel<gemm_deep_kernel<T, MT, MODE, EDGE>, (2 * kDeep + 1) * MT * kRowBytes>(p, timer, stream);
}

template <typename T, int MT>
static int launch_mode(int mode, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    if (mode == kSignal) return launch_t<T, MT, kSignal, false>(p, timer, stream);
    if (mode == kScatter) return launch_t<T, MT, kScatter, false>(p, timer, stream);
    return edge ? launch_t<T, MT, kPlain, true>(p, timer, stream) : launch_t<T, MT, kPlain, false>(p, timer, stream);
}

template <typename T>
static int launch_macro(int macro, int mode, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return macro == 64 ? launch_mode<T, 64>(mode, edge, p, timer, stream) : launch_mode<T, 128>(mode, edge, p, timer, stream);
}

int launch_gemm_deep(int macro, int mode, int dtype, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return dtype == FO_F16 ? launch_macro<_Float16>(macro, mode, edge, p, timer, stream)
                           : launch_macro<__bf16>(macro, mode, edge, p, timer, stream);
}

}  // namespace fo
