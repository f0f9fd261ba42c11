// The plain GEMM for a few rows of A (M <= 32): D = A . B^T where all the work is reading B once.
//
// A macro tile of 128 columns leaves most CUs without a tile (N = 4096: 32 of 128x128), and cutting
// those over K costs a second launch and a workspace.  Here a workgroup takes 16 rows of B, which is
// enough workgroups for most N, and its wavefronts share K between them in turns of 64; the sums meet
// in LDS, in the order of the wavefronts.
//
// Bound by what a CU loads per clock.  Loaded straight into the operand registers, where neighbouring
// lanes hold neighbouring rows, every lane is a line of its own to the address unit: 16 bytes per
// clock, 15 us for 16x4096x7168 bf16 however many loads are in flight.  So the turns are copied to LDS
// with the GEMM's copies, eight lanes to a line, and read from there as operands: the same row swizzle,
// but a ring of DEPTH turns per wavefront and no barrier, since a wavefront reads only what it copied.
// A is copied the same way (it is read once per workgroup, from the L2: for M <= 8 only its first
// eight rows), which is why more rows than 32 are left to the split tiles.  16x4096x7168: 10.6 us, 5.5
// TB/s of weights with the launch, against 15.8 as split tiles.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <atomic>

#include "fo_gemm_common.h"
#include "fo_internal.h"

namespace fo {

template <typename T>
struct Mfma16;
template <>
struct Mfma16<_Float16> {
    static __device__ __forceinline__ f32x4 run(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <>
struct Mfma16<__bf16> {
    static __device__ __forceinline__ f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

struct SkinnyParams {
    const void* A;
    const void* B;
    void* D;
    void* D2;   // also stored there, if not null
    int M, N, K;
};

// SLABS: copies of eight rows of A per turn (M <= 8 * SLABS).
template <typename T, int SLABS, int WAVES, int DEPTH>
__global__ void __launch_bounds__(64 * WAVES) skinny_kernel(const SkinnyParams p) {
    constexpr int MB = (SLABS + 1) / 2;                 // blocks of 16 rows of A
    constexpr int COPIES = 2 + SLABS;                   // 1 KiB copies per turn: 16 rows of B, 8 * SLABS of A
    constexpr int TURN = (2 + 2 * MB) * 1024;           // LDS bytes of a turn
    using frag = typename Mma<T>::frag;
    using out4 = typename Mma<T>::out4;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned char* ring = smem + wave * (DEPTH * TURN);
    const int n0 = blockIdx.x * 16;
    const unsigned row_bytes = (unsigned)p.K * 2u;
    // The descriptors end with the operands: rows beyond M or N, and (by an offset that lies beyond
    // either) the k beyond K, are written to LDS as zeros without touching memory.
    const __amdgpu_buffer_rsrc_t a = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, (int)((unsigned)p.M * row_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc((void*)p.B, 0, (int)((unsigned)p.N * row_bytes), 0x00020000);
    // A copy: lane l's 16 bytes land at row l / 8, chunk l % 8 of the slab and come from k-chunk
    // (l % 8) ^ swz(row); the slabs of a block differ in bit 3 of the row.
    const unsigned slab_row = lane >> 3;
    const unsigned chunk0 = ((lane & 7) ^ swz(slab_row)) * 16, chunk1 = ((lane & 7) ^ swz(slab_row + 8)) * 16;
    const unsigned row_b = ((unsigned)n0 + slab_row) * row_bytes, row_a = slab_row * row_bytes;
    auto copy = [&](int turn, int slot) {
        unsigned char* dst = ring + slot * TURN;
        const unsigned k = (unsigned)turn * 128u;
        const bool in0 = k + chunk0 < row_bytes, in1 = k + chunk1 < row_bytes;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const unsigned at = row_b + s * 8u * row_bytes + k + (s ? chunk1 : chunk0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (lds_void*)(dst + s * 1024), 16, (int)((s ? in1 : in0) ? at : 0xfffffff0u), 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < SLABS; ++s) {
            const unsigned at = row_a + s * 8u * row_bytes + k + ((s & 1) ? chunk1 : chunk0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a, (lds_void*)(dst + (2 + s) * 1024), 16, (int)(((s & 1) ? in1 : in0) ? at : 0xfffffff0u), 0, 0, 0);
        }
    };
    // Operands: lane l reads row l % 16, chunks 0, 2, 1, 3 (+ 4) of its lane group (see the GEMM).
    const int fr_row = lane & 15, fr_g = lane >> 4, fr_kc = (fr_g & 1) * 2 + (fr_g >> 1);
    int at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) at[h] = fr_row * kRowBytes + ((4 * h + fr_kc) ^ swz(fr_row)) * 16;

    f32x4 acc[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int turns = ((p.K + 63) / 64 + WAVES - 1) / WAVES;   // of every wavefront; turns beyond K are zeros
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) copy(d * WAVES + wave, d);
    for (int t0 = 0; t0 < turns; t0 += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            wait_vmcnt<(DEPTH - 1) * COPIES>();      // the oldest turn has landed
            __builtin_amdgcn_sched_barrier(0);
            const unsigned char* src = ring + d * TURN;
            frag fb[2], fa[2][MB];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                fb[h] = *(const frag*)(src + at[h]);
#pragma unroll
                for (int m = 0; m < MB; ++m) fa[h][m] = *(const frag*)(src + (2 + 2 * m) * 1024 + at[h]);
            }
            wait_lds_reads();                        // before the slot is copied to again
            __builtin_amdgcn_sched_barrier(0);
            copy((t0 + d + DEPTH) * WAVES + wave, d);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int m = 0; m < MB; ++m) acc[m] = Mfma16<T>::run(fb[h], fa[h][m], acc[m]);
        }
    wait_vmcnt<0>();
    __syncthreads();
    f32x4(*part)[MB][64] = (f32x4(*)[MB][64])smem;
#pragma unroll
    for (int m = 0; m < MB; ++m) part[wave][m][lane] = acc[m];
    __syncthreads();
    if ((int)threadIdx.x >= 64 * MB) return;
    const int m = threadIdx.x >> 6;
    f32x4 sum = part[0][m][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += part[w][m][lane];
    // a lane holds four consecutive n of one row
    const int row = 16 * m + (lane & 15), col = n0 + 4 * (lane >> 4);
    if (row >= p.M || col >= p.N) return;
    out4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (T)sum[r];
    const size_t off = (size_t)row * p.N + col;
    T* D = (T*)p.D;
    T* D2 = (T*)p.D2;
    if ((p.N & 3) == 0) {
        *(out4*)(D + off) = o;
        if (D2) *(out4*)(D2 + off) = o;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (col + r < p.N) {
                D[off + r] = o[r];
                if (D2) D2[off + r] = o[r];
            }
    }
}

template <typename T, int SLABS, int WAVES, int DEPTH>
static int launch_t(const SkinnyParams& p, const LaunchTimer& timer, hipStream_t stream) {
    constexpr int smem = WAVES * DEPTH * (2 + 2 * ((SLABS + 1) / 2)) * 1024;
    static_assert(smem <= 160 * 1024 && (DEPTH - 1) * (2 + SLABS) < 63);
    auto kern = skinny_kernel<T, SLABS, WAVES, DEPTH>;
    static std::atomic<unsigned long long> configured{0};   // once per device
    int dev = 0;
    FO_HIP(hipGetDevice(&dev));
    const unsigned long long bit = 1ull << (dev & 63);
    if (!(configured.load(std::memory_order_acquire) & bit)) {
        FO_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, smem));
        configured.fetch_or(bit, std::memory_order_release);
    }
    const dim3 grid((p.N + 15) / 16), block(64 * WAVES);
    if (timer.start) hipExtLaunchKernelGGL(kern, grid, block, smem, stream, timer.start, timer.stop, 0, p);
    else hipLaunchKernelGGL(kern, grid, block, smem, stream, p);
    FO_HIP(hipGetLastError());
    return FO_OK;
}

// Two turns in flight per wavefront are enough (more made no shape faster and those with more than one
// workgroup per CU slower); of these, and where A fills the LDS too, four wavefronts do better than eight.
// bf16, us with 4 / 8 wavefronts: 16x4096x7168 10.7 / 10.6, 8x1024x8192 8.4 / 7.0, 1x8192x3584 9.9 / 10.2,
// 3x6000x7000 14.2 / 15.2, 32x4096x7168 11.3 / 12.0.
template <typename T>
static int launch_dtype(const SkinnyParams& p, const LaunchTimer& timer, hipStream_t stream) {
    const bool four = p.N > 4096;
    if (p.M <= 8) return four ? launch_t<T, 1, 4, 2>(p, timer, stream) : launch_t<T, 1, 8, 2>(p, timer, stream);
    if (p.M <= 16) return four ? launch_t<T, 2, 4, 2>(p, timer, stream) : launch_t<T, 2, 8, 2>(p, timer, stream);
    return launch_t<T, 4, 4, 2>(p, timer, stream);
}

int launch_skinny(int dtype, int M, int N, int K, const void* A, const void* B, void* D, void* D2, const LaunchTimer& timer,
                  hipStream_t stream) {
    const SkinnyParams p{A, B, D, D2, M, N, K};
    return dtype == FO_F16 ? launch_dtype<_Float16>(p, timer, stream) : launch_dtype<__bf16>(p, timer, stream);
}

}  // namespace fo
