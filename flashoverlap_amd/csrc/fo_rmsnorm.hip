// RMSNorm and reorder+RMSNorm for gfx950.  Bound by HBM: every kernel reads a row once, keeps it in
// registers between the sum of squares and the scaling, and writes it once, in 128-bit accesses of
// whole cache lines.  Rows of up to 2048 elements take one 64-lane wavefront each, with a wavefront
// butterfly for the reduction (no LDS in it) and gamma staged in LDS once per workgroup while the rows'
// loads are in flight: held in registers beside the row it doubled the footprint, and the registers
// decide how many rows a SIMD has in flight.  Longer rows take a workgroup each; rows
// of more than 65536 elements a workgroup and two passes over memory.  The reorder
// variant gathers the row from the tile-permuted GEMM output: 16 consecutive
// lanes read one 256-byte row segment of a 128-wide tile, so every access is
// made of whole cache lines.  In the common case (rldn == 1, power-of-two tile,
// at most 64 tiles per row) the addresses take shifts only, and a wavefront that has a
// row to itself fetches one RA entry per lane and exchanges them, so the gather costs
// one small load instead of one per chunk.
//
// Arithmetic follows src/rmsnorm/rmsnorm.cuh:62-115 of the reference: fp32 sum
// of squares, scale = rsqrt(sum/dim + eps), the scaled value rounded to the
// storage type and then multiplied by gamma in the storage type (the product
// of two 16-bit floats is exact in fp32, so rounding it once equals the
// reference's half-precision multiply).  eps is a parameter here.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "fo_internal.h"

namespace fo {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <typename T>
struct Vec8;
template <>
struct Vec8<_Float16> {
    using type = f16x8;
};
template <>
struct Vec8<__bf16> {
    using type = bf16x8;
};

constexpr int kRowsPerBlock = 4;  // one wavefront per row; neighbouring rows read neighbouring tile segments
constexpr int kWideThreads = 256;  // rows too long for a workgroup's registers: one workgroup and two passes per row

// Ordinary loads, streaming (non-temporal) stores: the result is not read again here, and it
// must not displace the GEMM operands held in the memory-side cache.  Measured on 8192 x 4096
// against this choice (inside a step / one buffer pair back to back, 21.8 / 21.7 us as it is):
// non-temporal loads 21.8 / 25.5, ordinary stores 23.9 / 22.2; the other cache-policy bits on the
// stores (sc1, sc0 sc1, with and without nt) equal or slower.
template <typename V>
__device__ __forceinline__ V load_row_chunk(const V* p) {
    return *p;
}
template <typename V>
__device__ __forceinline__ void store_row_chunk(V v, V* p) {
    __builtin_nontemporal_store(v, p);
}

enum { kNormPlain = 0, kNormGather = 1, kNormGatherFast = 2 };

struct NormParams {
    int bs, dim, BM, BN, rldn;
    int log_bm, log_bn;  // kNormGatherFast only
    float eps;
};

// CH = 16-byte chunks per lane (dim <= CH * 512, CH <= 4).
template <typename T, int CH, int MODE>
__global__ void __launch_bounds__(64 * kRowsPerBlock) rmsnorm_kernel(const T* __restrict__ x0, const T* __restrict__ gamma,
                                                      T* __restrict__ out0, const int* __restrict__ RA,
                                                      const NormParams p) {
    using vec = typename Vec8<T>::type;
    extern __shared__ __attribute__((aligned(16))) unsigned char norm_smem[];   // dim * 2 bytes: gamma
    vec* lds_gamma = (vec*)norm_smem;
    const int lane = threadIdx.x & 63;
    const int row_of_wave = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    const bool live = row_of_wave < p.bs;
    const int row = live ? row_of_wave : p.bs - 1;   // a wavefront beyond the last row stays for the barrier, loading a row it never stores
    // blockIdx.y selects one of several independent [bs, dim] problems laid out back to back
    const T* __restrict__ x = x0 + (size_t)blockIdx.y * p.bs * p.dim;
    T* __restrict__ out = out0 + (size_t)blockIdx.y * p.bs * p.dim;

    const int dim = p.dim;
    const int nchunk = dim >> 3;
    vec xv[CH];
    if constexpr (MODE == kNormGatherFast) {
        // tiles of this row: RA[tile_row .. tile_row + ldn), ldn <= 64: one entry per lane
        const int ldn = dim >> p.log_bn;
        const int tile_row = (row >> p.log_bm) * ldn;
        const int in_row = row & (p.BM - 1);
        const int mine = RA[tile_row + (lane < ldn ? lane : 0)];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * 64 + lane;
            const int j = c << 3;
            const int s = __shfl(mine, (j >> p.log_bn) & 63, 64);  // all lanes take part in the exchange
            if (c < nchunk) {
                const size_t src = ((((size_t)s << p.log_bm) + in_row) << p.log_bn) + (j & (p.BN - 1));
                xv[k] = load_row_chunk((const vec*)(x + src));
            }
        }
    } else if constexpr (MODE == kNormGather) {
        const int ldn = dim / p.BN;
        const int tile_row = (row / p.BM) * ldn;
        const int in_row = row % p.BM;
        const int ld = p.rldn * p.BN;
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * 64 + lane;
            if (c < nchunk) {
                const int j = c << 3;
                const int s = RA[tile_row + j / p.BN];
                const size_t src = (size_t)((s / p.rldn) * p.BM + in_row) * ld + (s % p.rldn) * p.BN + j % p.BN;
                xv[k] = load_row_chunk((const vec*)(x + src));
            }
        }
    } else {
        const T* xr = x + (size_t)row * dim;
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * 64 + lane;
            if (c < nchunk) xv[k] = load_row_chunk((const vec*)(xr + (c << 3)));
        }
    }
    for (int c = threadIdx.x; c < nchunk; c += 64 * kRowsPerBlock) lds_gamma[c] = *(const vec*)(gamma + (c << 3));
    __syncthreads();
    if (!live) return;

    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        if (k * 64 + lane < nchunk) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = (float)xv[k][e];
                ss += f * f;
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const float scale = rsqrtf(ss / (float)dim + p.eps);
    // The row stays packed in its 16-bit form across the reduction; without this
    // the fp32 copies made for the sum of squares are kept alive too, which
    // doubles the register footprint and halves the waves per SIMD.
#pragma unroll
    for (int k = 0; k < CH; ++k) asm volatile("" : "+v"(xv[k]));

    T* orow = out + (size_t)row * dim;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        const int c = k * 64 + lane;
        if (c < nchunk) {
            const vec g = lds_gamma[c];
            vec o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const T y = (T)((float)xv[k][e] * scale);
                o[e] = (T)((float)y * (float)g[e]);
            }
            store_row_chunk(o, (vec*)(orow + (c << 3)));
        }
    }
}

// Longer rows: one workgroup per row, CH chunks per thread, the row in registers between the two
// passes over it, the wavefronts' partial sums added through LDS in a fixed order.  A long row held by one
// wavefront is a long serial chain (load it all, reduce, store it all) with few others beside it on
// the SIMD; four or eight wavefronts to the row have as many loads in flight and the next row's on
// their way meanwhile.  bf16, us, one wavefront / this kernel: reorder 8192x4096 21.9 / 20.7, 4096x5120
// 15.0 / 14.3, 512x8192 7.1 / 4.1, 16384x8192 95.3 / 93.3; plain 16384x8192 96.5 / 87.5 (6.1 TB/s), 4096x16384
// 51.0 / 46 (5.8), 2000x12288 18.1 / 15.7; against two passes over memory, which rows of more than 16384
// took: 1000x32768 28.4 / 20.4 (6.4), 500x65536 28.7 / 20.5.  Four wavefronts up to 6144 elements, eight
// above: at 8192 four are 2 % slower, at 5120 eight 8 % (half of them would have nothing to do).
template <typename T, int kTeamThreads, int CH, int MODE>
__global__ void __launch_bounds__(kTeamThreads) rmsnorm_team_kernel(const T* __restrict__ x0, const T* __restrict__ gamma,
                                                                  T* __restrict__ out0, const int* __restrict__ RA,
                                                                  const NormParams p) {
    using vec = typename Vec8<T>::type;
    __shared__ float part[kTeamThreads / 64];
    const int row = blockIdx.x, t = threadIdx.x;
    const T* __restrict__ x = x0 + (size_t)blockIdx.y * p.bs * p.dim;
    T* __restrict__ orow = out0 + (size_t)blockIdx.y * p.bs * p.dim + (size_t)row * p.dim;
    const int dim = p.dim, nchunk = dim >> 3;
    vec xv[CH], gv[CH];
    if constexpr (MODE == kNormPlain) {
        const T* xr = x + (size_t)row * dim;
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * kTeamThreads + t;
            if (c < nchunk) xv[k] = load_row_chunk((const vec*)(xr + (c << 3)));
        }
    } else {
        // where the tiles of this row lie: all lookups are issued before the first is used
        const int bm = MODE == kNormGatherFast ? row >> p.log_bm : row / p.BM;
        const int in_row = MODE == kNormGatherFast ? row & (p.BM - 1) : row % p.BM;
        const int tile_row = bm * (MODE == kNormGatherFast ? dim >> p.log_bn : dim / p.BN);
        int s[CH];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * kTeamThreads + t, j = c << 3;
            if (c < nchunk) s[k] = RA[tile_row + (MODE == kNormGatherFast ? j >> p.log_bn : j / p.BN)];
        }
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * kTeamThreads + t, j = c << 3;
            if (c >= nchunk) continue;
            const size_t src = MODE == kNormGatherFast
                                   ? ((((size_t)s[k] << p.log_bm) + in_row) << p.log_bn) + (j & (p.BN - 1))
                                   : (size_t)((s[k] / p.rldn) * p.BM + in_row) * (p.rldn * p.BN) + (s[k] % p.rldn) * p.BN + j % p.BN;
            xv[k] = load_row_chunk((const vec*)(x + src));
        }
    }
    // gamma comes from the L2: with few chunks it is asked for here, with many only when the row's registers are done with
    if constexpr (CH <= 2)
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int c = k * kTeamThreads + t;
            if (c < nchunk) gv[k] = *(const vec*)(gamma + (c << 3));
        }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < CH; ++k)
        if (k * kTeamThreads + t < nchunk) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = (float)xv[k][e];
                ss += f * f;
            }
        }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
    if ((t & 63) == 0) part[t >> 6] = ss;
    __syncthreads();
    float total = part[0];
#pragma unroll
    for (int w = 1; w < kTeamThreads / 64; ++w) total += part[w];
    const float scale = rsqrtf(total / (float)dim + p.eps);
#pragma unroll
    for (int k = 0; k < CH; ++k) asm volatile("" : "+v"(xv[k]));   // packed until here, as above
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        const int c = k * kTeamThreads + t;
        if (c >= nchunk) continue;
        if constexpr (CH > 2) gv[k] = *(const vec*)(gamma + (c << 3));
        vec o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const T y = (T)((float)xv[k][e] * scale);
            o[e] = (T)((float)y * (float)gv[k][e]);
        }
        store_row_chunk(o, (vec*)(orow + (c << 3)));
    }
}

// Rows longer than a workgroup keeps in registers (dim > 65536): one workgroup per row, two passes.
// The first pass sums the squares, the four wavefronts' partial sums meet in LDS (added in a fixed
// order), the second pass reads the row again (it is at most a few hundred KiB and still in the L2)
// and writes the result.  Same arithmetic per element as above; any dim that is a multiple of 8.
template <typename T, int MODE>
__global__ void __launch_bounds__(kWideThreads) rmsnorm_wide_kernel(const T* __restrict__ x0, const T* __restrict__ gamma,
                                                                  T* __restrict__ out0, const int* __restrict__ RA,
                                                                  const NormParams p) {
    static_assert(MODE == kNormPlain || MODE == kNormGather, "rows this long have more than 64 tiles");
    using vec = typename Vec8<T>::type;
    __shared__ float part[kWideThreads / 64];
    const int row = blockIdx.x;
    const T* __restrict__ x = x0 + (size_t)blockIdx.y * p.bs * p.dim;
    T* __restrict__ orow = out0 + (size_t)blockIdx.y * p.bs * p.dim + (size_t)row * p.dim;
    const int dim = p.dim, nchunk = dim >> 3;
    [[maybe_unused]] const int ldn = MODE == kNormGather ? dim / p.BN : 0;
    [[maybe_unused]] const int tile_row = MODE == kNormGather ? (row / p.BM) * ldn : 0;
    [[maybe_unused]] const int in_row = MODE == kNormGather ? row % p.BM : 0;
    auto chunk_at = [&](int c) -> const vec* {
        const int j = c << 3;
        if constexpr (MODE == kNormGather) {
            const int s = RA[tile_row + j / p.BN];
            return (const vec*)(x + (size_t)((s / p.rldn) * p.BM + in_row) * (p.rldn * p.BN) + (s % p.rldn) * p.BN + j % p.BN);
        } else {
            return (const vec*)(x + (size_t)row * dim + j);
        }
    };
    float ss = 0.f;
#pragma unroll 4
    for (int c = threadIdx.x; c < nchunk; c += kWideThreads) {
        const vec v = *chunk_at(c);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float f = (float)v[e];
            ss += f * f;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    float total = part[0];
#pragma unroll
    for (int w = 1; w < kWideThreads / 64; ++w) total += part[w];
    const float scale = rsqrtf(total / (float)dim + p.eps);
#pragma unroll 4
    for (int c = threadIdx.x; c < nchunk; c += kWideThreads) {
        const vec v = *chunk_at(c);
        const vec g = *(const vec*)(gamma + (c << 3));
        vec o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const T y = (T)((float)v[e] * scale);
            o[e] = (T)((float)y * (float)g[e]);
        }
        store_row_chunk(o, (vec*)(orow + (c << 3)));
    }
}

static int log2_exact(int v) {
    if (v <= 0 || (v & (v - 1))) return -1;
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
}

template <typename T, int MODE>
static int launch_wide(const void* x, const void* gamma, void* out, const int* RA, const NormParams& p, int nbatch,
                       const LaunchTimer& timer, hipStream_t stream) {
    const dim3 grid(p.bs, nbatch), block(kWideThreads);
    if (timer.start)
        hipExtLaunchKernelGGL((rmsnorm_wide_kernel<T, MODE>), grid, block, 0, stream, timer.start, timer.stop, 0,
                              (const T*)x, (const T*)gamma, (T*)out, RA, p);
    else
        hipLaunchKernelGGL((rmsnorm_wide_kernel<T, MODE>), grid, block, 0, stream, (const T*)x, (const T*)gamma, (T*)out,
                           RA, p);
    FO_HIP(hipGetLastError());
    return FO_OK;
}

template <typename T, int CH, int MODE>
static int launch_rows(const void* x, const void* gamma, void* out, const int* RA, const NormParams& p, int nbatch,
                       const LaunchTimer& timer, hipStream_t stream) {
    const dim3 grid((p.bs + kRowsPerBlock - 1) / kRowsPerBlock, nbatch), block(64 * kRowsPerBlock);
    const size_t smem = (size_t)p.dim * sizeof(T);
    if (timer.start)
        hipExtLaunchKernelGGL((rmsnorm_kernel<T, CH, MODE>), grid, block, smem, stream, timer.start, timer.stop, 0,
                              (const T*)x, (const T*)gamma, (T*)out, RA, p);
    else
        hipLaunchKernelGGL((rmsnorm_kernel<T, CH, MODE>), grid, block, smem, stream, (const T*)x, (const T*)gamma,
                           (T*)out, RA, p);
    FO_HIP(hipGetLastError());
    return FO_OK;
}

template <typename T, int W, int CH, int MODE>
static int launch_team(const void* x, const void* gamma, void* out, const int* RA, const NormParams& p, int nbatch,
                       const LaunchTimer& timer, hipStream_t stream) {
    const dim3 grid(p.bs, nbatch), block(W);
    if (timer.start)
        hipExtLaunchKernelGGL((rmsnorm_team_kernel<T, W, CH, MODE>), grid, block, 0, stream, timer.start, timer.stop, 0,
                              (const T*)x, (const T*)gamma, (T*)out, RA, p);
    else
        hipLaunchKernelGGL((rmsnorm_team_kernel<T, W, CH, MODE>), grid, block, 0, stream, (const T*)x, (const T*)gamma,
                           (T*)out, RA, p);
    FO_HIP(hipGetLastError());
    return FO_OK;
}

template <typename T, int MODE>
static int launch_t(const void* x, const void* gamma, void* out, const int* RA, const NormParams& p, int nbatch,
                    const LaunchTimer& timer, hipStream_t stream) {
    const int nchunk = p.dim / 8;
#define FO_NORM(KIND, ...) return launch_##KIND<T, __VA_ARGS__, MODE>(x, gamma, out, RA, p, nbatch, timer, stream)
    if (nchunk <= 64) FO_NORM(rows, 1);
    if (nchunk <= 128) FO_NORM(rows, 2);
    if (nchunk <= 256) FO_NORM(rows, 4);
    if (nchunk <= 512) FO_NORM(team, 256, 2);
    if (nchunk <= 768) FO_NORM(team, 256, 3);
    if (nchunk <= 1024) FO_NORM(team, 512, 2);
    if (nchunk <= 2048) FO_NORM(team, 512, 4);
    if (nchunk <= 4096) FO_NORM(team, 512, 8);
    if (nchunk <= 8192) FO_NORM(team, 512, 16);
#undef FO_NORM
    if constexpr (MODE == kNormGatherFast) return fail(FO_ERR_SHAPE, "fo_reorder_rmsnorm: dim=%d", p.dim);   // not selected for such rows
    else return launch_wide<T, MODE>(x, gamma, out, RA, p, nbatch, timer, stream);
}

template <typename T>
static int launch_dtype(const void* x, const void* gamma, void* out, const int* RA, const NormParams& p, int nbatch,
                        const LaunchTimer& timer, hipStream_t stream) {
    if (!RA) return launch_t<T, kNormPlain>(x, gamma, out, RA, p, nbatch, timer, stream);
    if (p.log_bm >= 0) return launch_t<T, kNormGatherFast>(x, gamma, out, RA, p, nbatch, timer, stream);
    return launch_t<T, kNormGather>(x, gamma, out, RA, p, nbatch, timer, stream);
}

int launch_rmsnorm(int dtype, const void* x, const void* gamma, void* out, int nbatch, int bs, int dim, int BM,
                   int BN, int rldn, const int* RA, float eps, hipStream_t stream) {
    const bool reorder = RA != nullptr;
    const char* who = reorder ? "fo_reorder_rmsnorm" : "fo_rmsnorm";
    // an event pair armed by fo_time_next_launch is this call's, whether or not it gets as far as a launch
    const LaunchTimer timer = t_launch_timer;
    t_launch_timer = LaunchTimer{};
    if (dtype != FO_F16 && dtype != FO_BF16) return fail(FO_ERR_ARG, "%s: dtype %d not fp16/bf16", who, dtype);
    if (bs == 0 || nbatch == 0) return FO_OK;
    if (nbatch < 0 || nbatch > 65535) return fail(FO_ERR_LIMIT, "%s: %d batches outside 0..65535", who, nbatch);
    if (!x || !gamma || !out) return fail(FO_ERR_ARG, "%s: null buffer", who);
    if (bs < 0 || dim <= 0) return fail(FO_ERR_SHAPE, "%s: bs=%d dim=%d", who, bs, dim);
    if (dim % 8) return fail(FO_ERR_SHAPE, "%s: dim=%d not a multiple of 8", who, dim);
    if ((long long)bs * dim * nbatch >= (1LL << 40)) return fail(FO_ERR_LIMIT, "%s: %lld elements", who, (long long)bs * dim * nbatch);
    if (((uintptr_t)x | (uintptr_t)gamma | (uintptr_t)out) & 15) return fail(FO_ERR_ARG, "%s: buffers must be 16-byte aligned", who);
    NormParams p{bs, dim, BM, BN, rldn, -1, -1, eps};
    if (reorder) {
        if (BM <= 0 || BN <= 0 || rldn <= 0) return fail(FO_ERR_ARG, "%s: BM=%d BN=%d rldn=%d", who, BM, BN, rldn);
        if (BN % 8 || dim % BN) return fail(FO_ERR_SHAPE, "%s: BN=%d must be a multiple of 8 that divides dim=%d", who, BN, dim);
        if (bs % BM) return fail(FO_ERR_SHAPE, "%s: bs=%d not a multiple of BM=%d", who, bs, BM);
        if (((long long)(bs / BM) * (dim / BN)) % rldn) return fail(FO_ERR_SHAPE, "%s: rldn=%d must divide the tile count", who, rldn);
        // (a wavefront that has a row to itself exchanges RA entries between its 64 lanes)
        if (rldn == 1 && dim <= 65536 && (dim > 2048 || dim / BN <= 64) && log2_exact(BM) >= 0 && log2_exact(BN) >= 0) {
            p.log_bm = log2_exact(BM);
            p.log_bn = log2_exact(BN);
        }
    }
    if (dtype == FO_F16) return launch_dtype<_Float16>(x, gamma, out, RA, p, nbatch, timer, stream);
    return launch_dtype<__bf16>(x, gamma, out, RA, p, nbatch, timer, stream);
}

}  // namespace fo
