// Internal declarations shared by the translation units of libfo_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/flashoverlap_hip.h"
#include "fo_plan.h"

namespace fo {

// Records the message returned by fo_last_error() and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define FO_HIP(expr)                                                                        \
    do {                                                                                    \
        hipError_t fo_e_ = (expr);                                                          \
        if (fo_e_ != hipSuccess)                                                            \
            return ::fo::fail(FO_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(fo_e_), \
                              __FILE__, __LINE__);                                          \
    } while (0)

int algo_tile(int algo, int* BM, int* BN, int* BK);

// fo_time_next_launch: a pair of events that the next GEMM or RMSNorm launch of this thread
// attaches to its own dispatch, so that the time between them is the kernel's, without the
// launch gaps an event pair recorded around the launch includes.  Taken by the launch that uses it.
// A call of several launches attaches `start` to the first and `stop` to the last.
struct LaunchTimer {
    hipEvent_t start = nullptr, stop = nullptr;
};
extern thread_local LaunchTimer t_launch_timer;

// fo_gemm.hip
int launch_gemm(const fo_gemm_call& c, hipStream_t stream, bool keep_d = true, fo_workspace_fn ask = nullptr, void* context = nullptr);
int gemm_workspace(const fo_gemm_call& c, size_t* bytes);
int gemm_rounds(int algo, int M, int N, int* per_round, int* last_first);
int raster_hint(int algo, int M, int N, int* hint);
int tune(const char* key, int value);

// fo_gemm_tall.hip, fo_gemm_deep.hip: the 256x128 macro tile; 64x64, and 128x128 with one workgroup to a CU
struct GemmParams;
int launch_gemm_deep(int macro, int mode, int dtype, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream);
int launch_gemm_tall(int mode, int dtype, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream);

// fo_skinny.hip: the plain GEMM for M <= kSkinnyRows.  bf16, us a call with 16 and 32 rows here, and with 33 and 64 in
// macro tiles (split over K but for the last shape), weights from the memory-side cache: 4096x7168 10.6 11.0 | 15.0 15.5,
// 8192x3584 10.6 11.5 | 14.8 15.3, 1024x8192 5.9 7.6 | 11.0 11.5, 3512x1408 4.9 4.8 | 6.6 6.5; weights from HBM: 13.0 16.1 |
// 16.8 17.4, 12.9 16.2 | 16.6 17.0, 11.0 14.3 | 11.9 12.6, 5.7 5.6 | 8.1 9.3.  The kernel grows with the rows (A is copied
// by every workgroup) and the macro tiles do not: at 32 rows the two meet where the weights come from HBM.
int launch_skinny(int dtype, int M, int N, int K, const void* A, const void* B, void* D, void* D2, int ld, bool across,
                  const LaunchTimer& timer, hipStream_t stream);   // across: D is stored transposed

// fo_splitk.hip: sums the parts of the split tiles and stores the tiles as the GEMM's epilogue would (stop: null, or
// an event of its end)
int launch_split_reduce(int mode, int dtype, int macro, const GemmParams& p, hipEvent_t stop, hipStream_t stream);

// fo_static.hip
int gemm_signal_static(int dtype, int algo, int M, int N, int K, int rLDN, const int* cseg, int G, const void* A,
                       const void* B, void* D, int* MM, const int* RA, int monitor, hipStream_t stream);

// fo_sync.hip
int launch_group_table(const int* cseg, int G, int T, int* table, int* start, hipStream_t stream);
int launch_wait(int that, int* addr, int* expired, hipStream_t stream);
int launch_wait_consume(const int* cseg, int G, int* MM, const void* src, void* dst, long long tile_elems,
                        int nslices, int slice_first, int slice_count, long long slice_stride, int* order_log,
                        int nblocks, int* expired, hipStream_t stream);
int launch_consume(const void* src, void* dst, size_t bytes, hipStream_t stream, int that = 0, int* addr = nullptr,
                   int nslices = 1, size_t dst_stride_bytes = 0, int policy = FO_COPY_AUTO, int* expired = nullptr);
int launch_wait_groups(const int* cseg, int first, int groups, int* MM, int* expired, hipStream_t stream);
int launch_consume_groups(const int* cseg, const int* gstart, int first, int groups, const void* src, void* dst,
                          long long tile_elems, int nslices, int slice_first, int slice_count, long long slice_stride,
                          int policy, size_t total_bytes, hipStream_t stream);
int set_wait_timeout_ms(int ms);
int wait_timeouts(int* count, int reset);

struct DeviceFacts {
    int wall_khz = 0;   // rate of wall_clock64()
    int cus = 0;
};
int device_facts(const DeviceFacts** out);   // of the current device

// fo_rmsnorm.hip
int launch_rmsnorm(int dtype, const void* x, const void* gamma, void* out, int nbatch, int bs, int dim, int BM,
                   int BN, int rldn, const int* RA, float eps, hipStream_t stream);

}  // namespace fo
