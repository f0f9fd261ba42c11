// The second half of a GEMM whose last tiles are split over K: adds the parts of every split tile up
// and stores the tile as the GEMM's epilogue stores the others (placement, delivery, signal).
//
// A problem of few tiles leaves most CUs idle, and the last round of any other that is not full does
// too: one workgroup walks all of K while its neighbours wait (128x4096x7168: 32 tiles of 128x128,
// 56 us, of which the weights are worth 8).  The parts are fp32, in the accumulators' own layout, and
// are added in the order of k, so a result does not depend on which part was finished first.  A
// kernel of its own and not the last workgroup to finish a tile: that one would read all parts of its
// tile alone (eight of 64 KiB at some 50 bytes per ns: 9 us), here every 16 rows of a wavefront's
// quadrant are a workgroup.  Bound by the memory-side cache the parts come from.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "fo_gemm_common.h"
#include "fo_internal.h"
#include "fo_raster.h"

namespace fo {

template <typename T, int MT, int MODE>
__global__ void __launch_bounds__(256) split_reduce_kernel(const GemmParams p) {
    constexpr int WT = MT / 2, NB = WT / 16;      // as in the GEMM: quadrant edge, 16x16 blocks per edge
    constexpr int VECS = NB * 64 / 256;           // four-float vectors per thread
    constexpr int PITCH = WT * 2 + 16;            // bytes of a row in LDS
    using out4 = typename Mma<T>::out4;
    __shared__ __attribute__((aligned(16))) unsigned char rows[16 * PITCH];

    const int tid = threadIdx.x;
    const int strip = blockIdx.x % NB, wave = blockIdx.x / NB % 4, tile = blockIdx.x / (4 * NB);
    const int wm = wave >> 1, wn = wave & 1;
    const TileCoord mt = macro_tile_at<MT, MT>(p, split_tile_pos(p, tile));
    if (mt.m * MT + wm * WT + 16 * strip >= p.M || mt.n * MT + wn * WT >= p.N) return;   // outside the matrix

    f32x4 sum[VECS];
    const f32x4* in = (const f32x4*)p.partial + partial_at(p, tile, 0, wave, NB * NB) + strip * NB * 64 + tid;
    const size_t next = (size_t)4 * NB * NB * 64;
#pragma unroll
    for (int v = 0; v < VECS; ++v) sum[v] = in[v * 256];
#pragma unroll 4
    for (int s = 1; s < p.splits; ++s)
#pragma unroll
        for (int v = 0; v < VECS; ++v) sum[v] += in[s * next + v * 256];

    int row0 = mt.m * MT + wm * WT, col0 = mt.n * MT + wn * WT, ld = p.N, slot = 0;
    bool deliver = p.D2 != nullptr, signal = false;
    if constexpr (MODE != kPlain) {
        slot = p.RA[((mt.m * MT + wm * WT) >> p.log_bm) * p.TN + ((mt.n * MT + wn * WT) >> p.log_bn)];
        row0 = (slot / p.rLDN) * p.BM + ((mt.m * MT + wm * WT) & (p.BM - 1));
        col0 = (slot % p.rLDN) * p.BN + ((mt.n * MT + wn * WT) & (p.BN - 1));
        ld = p.rLDN * p.BN;
        deliver = deliver && slot >= p.deliver_from;
        signal = !deliver;
    }
    row0 += 16 * strip;
    // a lane holds four consecutive n of one m: through LDS to whole row segments
#pragma unroll
    for (int v = 0; v < VECS; ++v) {
        const int at = v * 256 + tid, j = at >> 6, lane = at & 63;
        out4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (T)sum[v][r];
        *(out4*)(rows + (lane & 15) * PITCH + (16 * j + 4 * (lane >> 4)) * 2) = o;
    }
    __syncthreads();
    T* D = (T*)p.D;
    T* D2 = (T*)p.D2;
    if (tid < 2 * WT) {
        const int r = tid / (WT / 8), cc = tid % (WT / 8);
        const u32x4 v = *(const u32x4*)(rows + r * PITCH + cc * 16);
        int row = row0 + r;
        const int col = col0 + cc * 8;
        if constexpr (MODE == kScatter) row = p.RE[row];
        const size_t off = (size_t)row * ld + col;
        if constexpr (MODE == kPlain) {
            if (row < p.M && col < p.N) {
                store_edge_chunk(D + off, v, p.N - col);
                if (deliver) store_edge_chunk(D2 + off, v, p.N - col);
            }
        } else {
            if (signal) {   // write-through, see the GEMM's epilogue
                const __amdgpu_buffer_rsrc_t drsrc = __builtin_amdgcn_make_buffer_rsrc(p.D, 0, 0xffffffff, 0x00020000);
                __builtin_amdgcn_raw_buffer_store_b128(v, drsrc, (int)(off * 2), 0, 16);
            } else {
                *(u32x4*)(D + off) = v;
            }
            if (deliver) {
                if constexpr (MODE == kScatter) {
                    const int recv = receive_row(p, row, group_rows(p, slot));
                    if (recv >= 0) *(u32x4*)(D2 + (size_t)recv * ld + col) = v;
                } else {
                    *(u32x4*)(D2 + off) = v;
                }
            }
        }
    }
    if constexpr (MODE != kPlain) {
        if (!signal) return;   // (the same for the whole workgroup)
        // Acknowledged stores, then this strip counts itself; the last strip of a layout tile moves the
        // group's counter and leaves the strip count at zero for the next call.
        wait_vmcnt<0>();
        __syncthreads();
        if (tid == 0) {
            const int of_tile = ((wm * WT) >> p.log_bm) * (MT >> p.log_bn) + ((wn * WT) >> p.log_bn);
            int* arrived = p.arrived + 4 * tile + of_tile;
            const int strips = (p.BM / WT) * (p.BN / WT) * NB;
            if (__hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == strips - 1) {
                __hip_atomic_store(arrived, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const int group = p.gtable ? p.gtable[slot] : scan_group(p.cseg, slot);
                __hip_atomic_fetch_add(p.MM + group, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

template <typename T, int MT, int MODE>
static int launch_one(const GemmParams& p, hipEvent_t stop, hipStream_t stream) {
    const dim3 grid(p.split_tiles * 4 * (MT / 32)), block(256);
    if (stop) hipExtLaunchKernelGGL((split_reduce_kernel<T, MT, MODE>), grid, block, 0, stream, nullptr, stop, 0, p);
    else hipLaunchKernelGGL((split_reduce_kernel<T, MT, MODE>), grid, block, 0, stream, p);
    FO_HIP(hipGetLastError());
    return FO_OK;
}

template <typename T, int MT>
static int launch_t(int mode, const GemmParams& p, hipEvent_t stop, hipStream_t stream) {
    if (mode == kPlain) return launch_one<T, MT, kPlain>(p, stop, stream);
    return mode == kSignal ? launch_one<T, MT, kSignal>(p, stop, stream) : launch_one<T, MT, kScatter>(p, stop, stream);
}

int launch_split_reduce(int mode, int dtype, int macro, const GemmParams& p, hipEvent_t stop, hipStream_t stream) {
    if (dtype == FO_F16)
        return macro == 256 ? launch_t<_Float16, 256>(mode, p, stop, stream) : launch_t<_Float16, 128>(mode, p, stop, stream);
    return macro == 256 ? launch_t<__bf16, 256>(mode, p, stop, stream) : launch_t<__bf16, 128>(mode, p, stop, stream);
}

}  // namespace fo
