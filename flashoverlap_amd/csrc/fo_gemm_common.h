// Building blocks of the GEMM kernel in fo_gemm.hip: vector types, the MFMA wrappers, wait-count
// helpers, the LDS row swizzle, the launch parameters.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fo_internal.h"
#include "fo_raster.h"

namespace fo {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mma;
template <>
struct Mma<_Float16> {
    using frag = f16x8;
    using out4 = f16x4;
    static __device__ __forceinline__ void run(frag a, frag b, f32x4& c) {
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
    static __device__ __forceinline__ void clear(frag zeros, f32x4& c) {   // c = 0 x 0 + 0
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %1, 0" : "=a"(c) : "v"(zeros));
    }
};
template <>
struct Mma<__bf16> {
    using frag = bf16x8;
    using out4 = bf16x4;
    static __device__ __forceinline__ void run(frag a, frag b, f32x4& c) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
    static __device__ __forceinline__ void clear(frag zeros, f32x4& c) {   // c = 0 x 0 + 0
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %1, 0" : "=a"(c) : "v"(zeros));
    }
};

// The MFMAs above are opaque to the compiler: it does not know that their
// results become readable only some cycles after issue, and it inserts no wait
// states between one of them and an instruction that reads its accumulator.  So
// the accumulators are kept in the matrix-core register file (constraint "a")
// from the first MFMA to the epilogue, where they are read by this statement
// behind an explicit settle() — the compiler is then never asked to move an
// accumulator on its own (a copy it places right behind an MFMA reads the value
// from before that MFMA).
static __device__ __forceinline__ float acc_read(const float& a) {
    float v;
    asm("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));   // not volatile: free to be scheduled within the epilogue
    return v;
}
// The other direction, behind the last MFMA of a workgroup.
static __device__ __forceinline__ float acc_write(float v) {
    float a;
    asm("v_accvgpr_write_b32 %0, %1" : "=a"(a) : "v"(v));
    return a;
}
// More wait states than the longest MFMA needs before its result can be read.
static __device__ __forceinline__ void settle_mfma() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

constexpr int kRowBytes = kBK * 2;  // one panel row in LDS: 128 bytes = 8 chunks of 16

enum { kPlain = 0, kSignal = 1, kScatter = 2 };

// In the order in which a kernel wants them: the first read from each 64 bytes goes to memory, and what a plain GEMM
// reads lies in the first two lines, both touched while it starts (with the split's fields at the end, the 64x64 kernel met
// a third one in its last k-step: 512x1024x512 4.04 us, 3.86 so; 1024x1024x1024 5.59, 5.42; 64x7168x2048 8.71, 8.57).
struct GemmParams {
    const void* A;
    const void* B;
    void* D;      // null (signalling modes): every tile is delivered and stored there alone
    int M, N, K;
    int ld;       // plain: elements from one row of D to the next
    int GM, GN;   // macro-tile grid
    unsigned gn_magic;   // raster_magic(GN)
    // Tiles split over K: workgroups split_from .. split_from + split_tiles * splits - 1 compute a part
    // of `split_panels` panels of the macro tiles split_from .. split_from + split_tiles - 1 each and
    // leave it in `partial`; the reduction adds the parts up and stores the tiles (of 64x64 tiles, the
    // workgroup that finishes a tile's last part does).
    int split_from, split_tiles, splits, split_panels;
    int turn;     // 256x128 tiles: panels of K between the places where the XCDs begin, 0: all at the first
    float* partial;
    int* arrived;                               // strips of each layout tile that the reduction has stored; parts of each 64x64 tile that are in `partial`
    // delivery (null: none): tiles at slots >= deliver_from are stored there too, and not signalled
    void* D2;
    int deliver_from;
    int stream_deliver;                         // non-temporal stores there
    int BM, BN;   // layout tile
    int log_bm, log_bn;   // both edges are powers of two (128 or 256): shifts instead of divisions in the kernel
    int TN;       // N / BN
    int rLDN;
    const int* RA;
    const int* RE;
    const int* cseg;
    int G;
    const int* gtable;
    int* MM;
    int monitor;
    // delivery of a scatter
    const int* gstart;                          // first slot of every group
    int nslices, slice_first, slice_count;      // BM is a multiple of nslices
    int slice_rows;                             // rows of BN elements between the receive buffers
};

// Position of the macro tile of workgroup `tile` of the grid, and of split tile `index`: counted from
// split_from on if that is where a wave begins (the workgroups of its parts are shared out between the XCDs
// before they get here).
struct TilePos {
    int pos, by_column;   // for raster_tile
};
__device__ __forceinline__ TilePos whole_tile_pos(const GemmParams& p, int tile) {
    const int total = p.GM * p.GN;
    return {raster_pos(tile, total), raster_whole(total)};
}
__device__ __forceinline__ TilePos split_tile_pos(const GemmParams& p, int index) {
    return p.split_from % kWave ? whole_tile_pos(p, p.split_from + index) : TilePos{p.split_from + index, p.GM * p.GN};
}
template <int MTM, int MTN>
__device__ __forceinline__ TileCoord macro_tile_at(const GemmParams& p, TilePos at) {
    if constexpr (MTM > MTN) return raster_tile<kGroupM / 2, kUnitN * 2>(at.pos, p.GM, p.GN, p.gn_magic, at.by_column);
    else return raster_tile(at.pos, p.GM, p.GN, p.gn_magic, at.by_column);
}

// Where a part of a split tile lies in `partial`: [tile][split][wave][block i * NB + j][lane] vectors of
// four floats, i.e. as the accumulators lie in the wavefronts; every access is a contiguous KiB.
__device__ __forceinline__ size_t partial_at(const GemmParams& p, int tile, int split, int wave, int blocks) {
    return ((size_t)(tile * p.splits + split) * 4 + wave) * blocks * 64;
}

// Scatter, delivered tiles.  A group's rows are cut into nslices equal parts (fo_wait_consume).
struct GroupRows {
    int first, part;   // first row of a group in the permuted view, rows of a slice
};
__device__ __forceinline__ GroupRows group_rows(const GemmParams& p, int slot) {
    const int g = p.gtable[slot];
    return {p.gstart[g] << p.log_bm, (p.cseg[g] << p.log_bm) / p.nslices};
}
// The row of the receive buffers that row q of the permuted view goes to, -1 if this call keeps no
// buffer for its slice.  The row map permutes rows inside a group; a row that it sends out of its
// tile's group looks its own group up.
__device__ __forceinline__ int receive_row(const GemmParams& p, int q, GroupRows r) {
    if ((unsigned)(q - r.first) >= (unsigned)(r.part * p.nslices)) r = group_rows(p, q >> p.log_bm);
    const unsigned in_group = (unsigned)(q - r.first);
    const int slice = (int)(in_group / (unsigned)r.part) - p.slice_first;
    if (slice < 0 || slice >= p.slice_count) return -1;
    return slice * p.slice_rows + r.first / p.nslices + (int)(in_group % (unsigned)r.part);
}

typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt immediate of the gfx9 family: vmcnt in bits [3:0] and [15:14],
// expcnt [6:4], lgkmcnt [11:8]; 63 / 7 / 15 mean "do not wait".
constexpr int waitcnt_imm(int vm, int lgkm) {
    return (vm & 0xF) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm & 0xF) << 8);
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(N, 15));
}
__device__ __forceinline__ void wait_lds_reads() { __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0)); }

// The reference's linear scan over cSeg (src/overlap/gemm_with_signal.h:188-193).
__device__ __forceinline__ int scan_group(const int* cseg, int slot) {
    int bound = cseg[0];
    int g = 0;
    while (bound <= slot) {
        ++g;
        bound += cseg[g];
    }
    return g;
}

// Row swizzle shared by the copy and the fragment reads: LDS chunk (row, cc)
// holds k-chunk cc ^ swz(row).  Any 8 (or, two rows per 256 bytes, any 16)
// consecutive rows then hit distinct banks when they read the same k-chunk.
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// Eight elements of a row of which `left` lie inside the matrix, at an address that is a multiple of
// the element size only (N need not be a multiple of 8): one 16-byte store where all eight do - the
// compiler knows that global memory takes it at any alignment - and the elements one by one where
// the row ends.
template <typename T>
__device__ __forceinline__ void store_edge_chunk(T* to, u32x4 v, int left) {
    struct __attribute__((packed, aligned(2))) chunk {
        u32x4 v;
    };
    if (left >= 8) {
        ((chunk*)to)->v = v;
        return;
    }
    const T* e = (const T*)&v;
#pragma unroll
    for (int k = 0; k < 7; ++k)
        if (k < left) to[k] = e[k];
}

template <int N>
using template_int = std::integral_constant<int, N>;

// f(integral_constant<0>) ... f(integral_constant<N-1>)
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(template_int<N - 1>{});
    }
}

}  // namespace fo
