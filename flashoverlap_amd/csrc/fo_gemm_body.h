// The signalling GEMM's kernel body for gfx950 (MI355X): D = A . B^T, A [M,K], B [N,K], both with
// K contiguous, 16-bit inputs (fp16 / bf16), fp32 accumulation on MFMA.
//
// One workgroup of 4 wavefronts computes one MTM x MTN macro tile (256 x 256, or
// 256 x 128, 128 x 128 or 64 x 64 where those are too few to fill the GPU); each wavefront
// owns an (MTM/2) x (MTN/2) quadrant as 16 x 16 blocks of v_mfma_f32_16x16x32,
// accumulators in AGPRs.  The 16x16x32
// form reads and writes a quarter of the accumulator registers per flop of the
// 32x32x16 form (the k-reduction of 32 happens inside the instruction); the
// chip runs this kernel at its power limit, and the kernel measured 3-4 %
// faster with it.  The MFMAs are issued through inline assembly with the
// accumulators pinned to AGPRs: with the compiler builtin the register
// allocator moved 16x16 accumulators between the two register files inside
// the main loop.  The order of the main loop's instructions is therefore
// written out slot by slot in the source and fenced, not left to the scheduler.
//
// Main loop: A and B panels of 64 k-elements stream HBM -> LDS with
// buffer_load_dwordx4 ... lds (no register staging) into two A and three B panel
// slots (all of the 160 KiB of LDS at 256 x 256): the A and B panels of the
// k-step being multiplied, those of the next one, and one free slot.  A panel
// row is 128 bytes, so every copy instruction fetches eight whole cache lines:
// the L2 serves one request per channel per clock whatever its size, and at
// this tile size the kernel sits at the edge of that request rate, so half-line
// requests cost a quarter of the throughput.  The 16-byte chunks of a row are
// XOR-swizzled by row so the ds_read_b128 fragment reads are bank-conflict
// free.  A k-step of 64 is two half steps of 64 MFMAs, each over half the rows
// of blocks and walked column by column, with the two MFMAs that an
// accumulator gets from the panel (k halves 0 and 1) issued back to back: the
// second then takes the running sum from inside the matrix core instead of
// from the register file, which lowers the power per flop and with it raises
// the clock the power limit allows.  All B fragments of the panel stay in
// registers for the whole k-step and are replaced, column by column, by those
// of the next panel during the second half step; the A fragments of the
// second half step are read during the first, so all reads of a panel are out
// by the middle of its k-step, where the workgroup barrier that releases the
// panel's two slots sits.  The free slot lets the copies of B(p+2) go out in
// the first half of k-step p and those of A(p+2) in the second half, one
// every few MFMAs, with more than a k-step to land, which is what the kernel
// needs when its operands come from HBM and not from the memory-side cache.
// There is one barrier per k-step.
//
// Epilogue: the quadrant goes through LDS in strips of 32 rows so that every
// global store instruction writes four whole 256-byte row segments, either to
// the natural row-major D (plain GEMM) or to slot RA[tile] of the
// tile-permuted layout, optionally with the row index mapped through RE
// (scatter).  Then the signal: after every wavefront's stores have been
// acknowledged and the workgroup has met at a barrier, one lane per layout
// tile bumps the tile's group counter with an agent-scope atomic.  The tile
// stores are agent-scope write-through stores (sc1), the instruction the
// compiler emits for an agent-scope atomic store: once s_waitcnt vmcnt(0)
// returns they have been performed at agent scope, so nothing dirty is left in
// this XCD's L2 for a release to write back, and the counter atomic can be a
// relaxed one.  (The release-ordered form, cached stores or not, is kept as a
// tuning knob: its buffer_wbl2 costs 3-10 % of a short-K GEMM.)  The plain
// GEMM is the same kernel with the signalling compiled out.
//
// Delivery: the epilogue can store a tile a second time, to where the consumer would have copied it, and
// leave its counter alone.  The second store of a strip comes from the same registers; what it saves is the
// read of C, the copy's traffic beside the GEMM and one wait and one copy launch per group (4096x4096x4096 fp16 in
// 16 groups: the overlapped call and its norm 239 -> 117 us; 1024x1024x1024 in 16: 135 -> 14;
// 128x4096x7168 bf16 in one: 65.6 -> 61.1; plain GEMM 16x4096x7168 with its bulk
// copy: 63.1 -> 58.8).  Of the two copies of a call that delivers every tile, D itself is what nobody reads next: stored
// past the caches it leaves them to the other one (write-through / so, with the norm: 16384x8192x1024 386 / 371 us, 3840x7808x880
// 86 / 78, 7424x6016x640 116 / 111, plain 8191x8184x512 with its bulk copy 187 / 161; in one round, level).  A caller that keeps only
// the other one passes no D.  One that does read C next, in its copy's place, pays up to 5 % where C would have stayed in a cache (plain
// call with a norm of C, write-through / so: 7424x6016x640 92.5 / 97.0, 3840x7808x880 75.0 / 78.6, 8192x4096x1024 87.4 / 88.9,
// 4096x4096x4096 109.5 / 110.5) and gains with a larger one (8191x8184x512 136 / 134, 16384x8192x1024 354 / 323).
//
// Semantics follow the reference epilogues src/overlap/gemm_with_signal.h:145-201
// and src/overlap/gemm_with_scatter.h:146-196; the kernel itself shares nothing
// with the reference's MUTlass mainloop.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "fo_gemm_common.h"
#include "fo_raster.h"

namespace fo {

// LDS of the panel slots: `depth` of A and one more of B.
constexpr int ring_bytes(int mtm, int mtn, int depth) { return (depth * mtm + (depth + 1) * mtn) * kRowBytes; }

// STORE: 0 cached, 1 write-through tile stores; REL: 0 release atomic, 1 relaxed atomic.
// EDGE (plain GEMM only): M and N are arbitrary; the rows and columns of a macro tile that lie
// outside the matrix are computed on zeros and not stored.
// DEPTH: panels ahead of the one being multiplied that are in LDS or on their way there.
template <typename T, int MTM, int MTN, int MODE, int STORE, int REL, bool EDGE, int DEPTH = 2>
__device__ __forceinline__ void gemm_body(const GemmParams& p) {
    static_assert(!EDGE || MODE == kPlain, "only the plain GEMM takes shapes that are not multiples of the layout tile");
    constexpr int WM = MTM / 2, WN = MTN / 2;    // wave quadrant
    constexpr int NBM = WM / 16, NBN = WN / 16;  // its 16x16 MFMA blocks
    constexpr int NH = NBM / 2;                  // rows of blocks per half step
    constexpr int PANEL_A = MTM * kRowBytes, PANEL_B = MTN * kRowBytes;
    constexpr int LOADS_A = MTM / 32, LOADS_B = MTN / 32;        // wave-wide 1 KiB copies per wave per panel
    constexpr int B_RING = DEPTH * PANEL_A;  // where the B panels' slots begin
    constexpr int BLK = 16 * kRowBytes;      // LDS bytes between 16-row blocks
    using frag = typename Mma<T>::frag;
    using out4 = typename Mma<T>::out4;

    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

    static_assert(2 * 4 * 32 * (WN * 2 + 16) <= ring_bytes(MTM, MTN, DEPTH), "epilogue strips must fit in the panel slots");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    const int K = p.K;
    const int NPK = (K + kBK - 1) / kBK;   // panels of the whole K, the last one possibly partial
    // A split tile: this workgroup multiplies NP panels from kt0 on.  The workgroups of an XCD
    // (blockIdx.x % 8; split_from is a multiple of 8) get consecutive numbers, split by split, so that
    // they work on one range of k and share its panels in their L2.
    int tile = blockIdx.x, kt0 = 0, NP = NPK, part = -1;
    TilePos at_tile;
    if (MTM == MTN && tile >= p.split_from) {
        const unsigned q = tile - p.split_from, all = p.split_tiles * p.splits, even = all & ~(kXcds - 1);
        const unsigned at = q < even ? (q & (kXcds - 1)) * (even / kXcds) + q / kXcds : q;
        part = at / (unsigned)p.split_tiles;
        tile = at - part * p.split_tiles;
        at_tile = split_tile_pos(p, tile);
        kt0 = part * p.split_panels;
        NP = min(p.split_panels, NPK - kt0);
    } else {
        at_tile = whole_tile_pos(p, tile);
    }
    const TileCoord mt = macro_tile_at<MTM, MTN>(p, at_tile);
    // One round of 256x128 tiles (turn_panels in fo_plan.h): the XCDs begin at eight places of K, panel kt of a workgroup is panel
    // kt + turn, and behind the last one comes the first.  Inside an XCD all begin at the same place, for they share panels in its L2,
    // and neighbours three eighths apart (one eighth: 1.026 times as long on 70 shapes, bf16, operands from HBM).  Parts of split tiles
    // begin at different places as it is, and several rounds of 256x256 tiles lose (8192x4096x7168 with its norm 348 / 357 us).
    int turn = 0;
    if constexpr (MTM != MTN) turn = (int)(blockIdx.x * 3u % kXcds) * p.turn;
    int k_first = kt0 + turn;   // panel kt of this workgroup is panel kt + k_first of K (the main loop turns back to the first)
    // M and N are multiples of the layout tile, not necessarily of the macro
    // tile: the last row or column of macro tiles may be half inside.  Such a
    // workgroup runs the full main loop (the waves of the outer half re-read the
    // panel rows of the inner half, so nothing outside the operands is touched)
    // and only the quadrants inside are stored and signalled.  EDGE: M and N are
    // arbitrary; the panel rows beyond the matrix are zero-filled by the
    // hardware (see the copy addressing below) and only the rows and columns
    // inside the matrix are stored.
    const int valid_m = min(MTM, p.M - mt.m * MTM), valid_n = min(MTN, p.N - mt.n * MTN);
    const bool live = wm * WM < valid_m && wn * WN < valid_n;                          // this wave's quadrant

    // ---- where this wavefront's quadrant goes -------------------------------
    // row0/col0/ld describe the destination of quadrant element (0,0) in a
    // row-major view; rows are consecutive in that view (before RE).  In the
    // signalling modes they follow from the slot of the quadrant's layout tile.
    // The slots (this wave's, and in the lanes that will signal that of "their"
    // layout tile) are fetched here, ahead of the first panel copies, but looked at
    // only behind the prologue's barrier, when they have long arrived: nothing may
    // stand between the start of the kernel and the issue of those copies.  What
    // depends on the slots (group, remapped rows) is fetched there too, under the
    // first k-steps.
    int row0 = mt.m * MTM + wm * WM, col0 = mt.n * MTN + wn * WN, ld = p.ld;
    int sig_slot = 0, sig_group = -1;   // -1: a lane without a layout tile inside the matrix stays out of the signal
    [[maybe_unused]] int quad_slot = 0;
    [[maybe_unused]] bool sig_lane = false;
    if constexpr (MODE != kPlain) {
        const int tiles_n = MTN >> p.log_bn;          // layout tiles per macro tile, N
        const int tiles_m = MTM >> p.log_bm;
        // (a layout tile may also be larger than the macro tile, if nothing is signalled: no lane then has one to signal)
        if (live) quad_slot = p.RA[((mt.m * MTM + wm * WM) >> p.log_bm) * p.TN + ((mt.n * MTN + wn * WN) >> p.log_bn)];
        const int sig_m = tiles_n == 2 ? tid >> 1 : tid, sig_n = tiles_n == 2 ? tid & 1 : 0;   // tiles_n is 1 or 2
        sig_lane = tid < tiles_m * tiles_n && (sig_m << p.log_bm) < valid_m && (sig_n << p.log_bn) < valid_n;
        if (sig_lane) sig_slot = p.RA[(mt.m * tiles_m + sig_m) * p.TN + mt.n * tiles_n + sig_n];
    }
    [[maybe_unused]] int re_lo = 0, re_hi = 0;   // scatter: the remapped destination rows of this quadrant
    [[maybe_unused]] int dl_lo = -1, dl_hi = -1; // scatter: their rows in the receive buffers, -1: not delivered
    [[maybe_unused]] GroupRows tile_group{0, 1};
    bool deliver = MODE == kPlain && p.D2 != nullptr;
    auto resolve_destination = [&]() {
        if constexpr (MODE != kPlain) {
            const int s = __builtin_amdgcn_readfirstlane(quad_slot);
            row0 = (s / p.rLDN) * p.BM + ((mt.m * MTM + wm * WM) & (p.BM - 1));
            col0 = (s % p.rLDN) * p.BN + ((mt.n * MTN + wn * WN) & (p.BN - 1));
            ld = p.rLDN * p.BN;
            // a delivered tile is not signalled: nobody waits for it
            if (sig_lane && !(p.D2 && sig_slot >= p.deliver_from))
                sig_group = p.gtable ? p.gtable[sig_slot] : scan_group(p.cseg, sig_slot);
            deliver = p.D2 && s >= p.deliver_from;
        }
        // Scatter: one or two remapped rows per lane, handed round between the lanes in the epilogue.
        if constexpr (MODE == kScatter) {
            re_lo = p.RE[row0 + (lane < WM ? lane : 0)];
            if constexpr (WM > 64) re_hi = p.RE[row0 + 64 + lane];
            if (deliver) tile_group = group_rows(p, __builtin_amdgcn_readfirstlane(quad_slot));
        }
    };

    // ---- HBM -> LDS copy addressing ------------------------------------------
    // One copy instruction moves 1 KiB = 8 panel rows of 128 bytes: lane l's 16
    // bytes land at the LDS base + 16*l, i.e. row l/8, chunk l%8 of the slab, and
    // are fetched from k-chunk (l%8) ^ swz(row).  Buffer addressing: the operand
    // is the buffer, the wave-uniform part of the offset (panel row, slab, k)
    // lives in a scalar register and only the constant per-lane part in a vector
    // register, so a copy costs no vector ALU work.  Slabs alternate in bit 3 of
    // the row number, hence two per-lane offsets.
    const int cp_row = lane >> 3;
    const int cp_off0 = (cp_row * K + ((lane & 7) ^ swz(cp_row)) * 8) * 2;       // even slabs
    const int cp_off1 = (cp_row * K + ((lane & 7) ^ swz(cp_row + 8)) * 8) * 2;   // odd slabs
    // K need not be a multiple of the panel depth.  In the last, partial panel the
    // lanes whose k-chunk lies beyond K take a per-lane offset outside the buffer's
    // range instead: the hardware then fetches nothing for them and writes zeros to
    // their LDS bytes, so the panel is zero-padded and the main loop needs no k
    // mask.  The range (2 GiB, checked against the operand sizes on the host) only
    // has to separate that one offset from the real ones.
    const int k_rest = kt0 + NP == NPK ? K % kBK : 0;
    constexpr int kOutOfRange = (int)0x80000000u;
    int tail_off0 = cp_off0, tail_off1 = cp_off1;
    if (k_rest) {
        if (((lane & 7) ^ swz(cp_row)) * 8 >= k_rest) tail_off0 = kOutOfRange;
        if (((lane & 7) ^ swz(cp_row + 8)) * 8 >= k_rest) tail_off1 = kOutOfRange;
    }
    int vo0 = cp_off0, vo1 = cp_off1;   // the offsets in use: the tail pair for the last panel
    const int range = k_rest ? kOutOfRange : (int)0xffffffffu;
    // EDGE: the hardware checks only the per-lane part of an offset against the descriptor's range.
    // So the descriptor of an operand starts at the macro tile's first row and ends with the operand,
    // the row inside the tile goes into the per-lane part (one addition per copy) and only the k
    // position stays scalar: a lane whose row lies beyond the matrix is then out of range, fetches
    // nothing and gets zeros, whatever M and N are.
    const __amdgpu_buffer_rsrc_t rsrcA =
        EDGE ? __builtin_amdgcn_make_buffer_rsrc((char*)p.A + (size_t)mt.m * MTM * K * 2, 0,
                                                 (int)((unsigned)(p.M - mt.m * MTM) * (unsigned)K * 2u), 0x00020000)
             : __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, range, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcB =
        EDGE ? __builtin_amdgcn_make_buffer_rsrc((char*)p.B + (size_t)mt.n * MTN * K * 2, 0,
                                                 (int)((unsigned)(p.N - mt.n * MTN) * (unsigned)K * 2u), 0x00020000)
             : __builtin_amdgcn_make_buffer_rsrc((void*)p.B, 0, range, 0x00020000);
    const unsigned baseA = EDGE ? (unsigned)(wave * (LOADS_A * 8)) * (unsigned)K * 2u
                                : (unsigned)(mt.m * MTM + ((wave * (LOADS_A * 8)) & (valid_m - 1))) * (unsigned)K * 2u;
    const unsigned baseB = EDGE ? (unsigned)(wave * (LOADS_B * 8)) * (unsigned)K * 2u
                                : (unsigned)(mt.n * MTN + ((wave * (LOADS_B * 8)) & (valid_n - 1))) * (unsigned)K * 2u;
    const unsigned slab_bytes = 8u * (unsigned)K * 2u;    // bytes between consecutive slabs
    const int lds_cpA = wave * (LOADS_A * 1024), lds_cpB = wave * (LOADS_B * 1024);   // this wave's first slab in a panel

    // The LDS holds two rings, DEPTH slots of A panels and behind them DEPTH + 1 of B panels; panel kt lives in
    // slot kt % DEPTH of the one and kt % (DEPTH + 1) of the other.  `slot` is the byte offset of
    // the receiving slot; the copies of a unit (an A or a B panel) are issued in two halves.
    auto issue_unit = [&](int kt, int slot, auto isb_c, auto half_c) {
        constexpr bool ISB = decltype(isb_c)::value;
        constexpr int H = decltype(half_c)::value;
        constexpr int LOADS = ISB ? LOADS_B : LOADS_A;
        unsigned char* dst = smem + slot + (ISB ? lds_cpB : lds_cpA);
        const unsigned koff = (unsigned)(k_first + kt) * (kBK * 2);
#pragma unroll
        for (int j = H * (LOADS / 2); j < (H + 1) * (LOADS / 2); ++j) {
            const int voff = (j & 1) ? vo1 : vo0;   // LOADS*8 is a multiple of 16: slab parity = j parity
            const unsigned rows = (ISB ? baseB : baseA) + j * slab_bytes;   // the slab's first row, in bytes
            if constexpr (ISB)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcB, (lds_void*)(dst + j * 1024), 16, EDGE ? (int)((unsigned)voff + rows) : voff,
                                                         (int)(EDGE ? koff : rows + koff), 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcA, (lds_void*)(dst + j * 1024), 16, EDGE ? (int)((unsigned)voff + rows) : voff,
                                                         (int)(EDGE ? koff : rows + koff), 0, 0);
        }
    };
    std::false_type unit_a;
    std::true_type unit_b;

    // ---- LDS -> register fragment addressing ----------------------------------
    // MFMA 16x16x32 operand: lane l supplies row l%16 and the 8 k-values of lane
    // group l/16.  Which 8 of the k half's 32 a group takes is free as long as A
    // and B agree; groups 0..3 take the 16-byte chunks 0, 2, 1, 3.  The LDS
    // serves lanes l and l+32 in the same pass: this way the two read
    // neighbouring chunks of one row, which the row swizzle keeps on different
    // banks (chunks 0 and 2 of the same rows would collide two ways).
    const int fr_row = lane & 15, fr_g = lane >> 4;
    const int fr_kc = (fr_g & 1) * 2 + (fr_g >> 1);
    const int a_lane = (wm * WM + fr_row) * kRowBytes;
    const int b_lane = (wn * WN + fr_row) * kRowBytes;
    int ko[2];   // chunk offset of each k half (k 0..31, 32..63)
#pragma unroll
    for (int h = 0; h < 2; ++h) ko[h] = ((4 * h + fr_kc) ^ swz(fr_row)) * 16;

    f32x4 acc[NBM][NBN];   // cleared in the prologue, while the first panels are on their way

    // Fragments of the two k halves of a panel.  The B blocks of both halves stay in registers for
    // the whole k-step; the A blocks come in two sets, rows of blocks 0..NH-1 for the first half of
    // the k-step and NH..NBM-1 for the second.
    frag fa[2][NBM], fb[2][NBN];   // [k half][block]

    // One copy instruction (slab j of the A or B unit of panel kt) into slot `slot`.
    auto issue_one = [&](int kt, int slot, auto isb_c, auto j_c) {
        constexpr bool ISB = decltype(isb_c)::value;
        constexpr int j = decltype(j_c)::value;
        unsigned char* dst = smem + slot + (ISB ? lds_cpB : lds_cpA);
        const unsigned koff = (unsigned)(k_first + kt) * (kBK * 2);
        const int voff = (j & 1) ? vo1 : vo0;
        const unsigned rows = (ISB ? baseB : baseA) + j * slab_bytes;
        if constexpr (ISB)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcB, (lds_void*)(dst + j * 1024), 16, EDGE ? (int)((unsigned)voff + rows) : voff,
                                                     (int)(EDGE ? koff : rows + koff), 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcA, (lds_void*)(dst + j * 1024), 16, EDGE ? (int)((unsigned)voff + rows) : voff,
                                                     (int)(EDGE ? koff : rows + koff), 0, 0);
    };
    // One fragment read.
    auto read_a = [&](int slot_a, int h, int i) { fa[h][i] = *(const frag*)(smem + slot_a + ko[h] + a_lane + i * BLK); };
    auto read_b = [&](int slot_b, int h, int j) { fb[h][j] = *(const frag*)(smem + slot_b + ko[h] + b_lane + j * BLK); };

    // One k-step on panel kt (at DEPTH 2; of a deeper ring the copies are those of panel kt+DEPTH).
    // A(kt) sits in slot sa, the units of panel kt+1 in na and nb (landed or landing), sp is the free slot of the B ring; the B fragments of panel kt and the A fragments of its
    // first NH rows of blocks are in registers, or on their way there, on entry.
    //
    // The two MFMAs that an accumulator gets from a panel (k halves 0 and 1) are issued back to
    // back: the second then takes the running sum from inside the matrix core instead of from the
    // register file, and a loop of bare MFMAs in this order runs 5-7 % faster at the chip's power
    // limit than one that visits every accumulator once per k half.  The order is column by
    // column (B block j with the NH rows of the half step, both k halves each), which is what
    // lets the B fragments be replaced one column at a time:
    //   half step 0: rows 0..NH-1.  Reads the A fragments of rows NH..NBM-1; copies B(kt+2) to the
    //     free slot.  All reads of panel kt are issued by its end, so its two slots are handed over at
    //     the barrier in the middle of the k-step.
    //   half step 1: rows NH..NBM-1.  Reads the first A fragments of panel kt+1 and, behind the last
    //     MFMA of column j, the B fragments j of panel kt+1 into the registers that column just
    //     left; copies A(kt+2) to slot sa.
    // LDS reads return in order.  Half step 0 therefore starts column j as soon as at most
    // 2(NBN-1-j) reads younger than B fragments j are outstanding, plus its own reads issued so far.
    // NEXT: panel kt+1 exists.  C2: panel kt+DEPTH exists.
    constexpr int COL = 2 * NH;          // MFMAs per column of a half step
    constexpr int NS = COL * NBN;        // MFMAs per half step
    auto half_step = [&](auto hs_c, int kt, int slot_reads_a, int slot_next_b, int slot_copy, auto next_c, auto c2_c) {
        constexpr int hs = decltype(hs_c)::value;
        constexpr bool NEXT = decltype(next_c)::value;
        constexpr bool C2 = decltype(c2_c)::value;
        constexpr int i0 = hs * NH;
        constexpr int CP_EVERY = NS / (hs ? LOADS_A : LOADS_B);   // one copy every so many MFMAs
        static_for<NS>([&](auto s_c) {
            constexpr int sl = decltype(s_c)::value;
            constexpr int j = sl / COL, w = sl % COL, h = w & 1;
            constexpr int r = (j & 1) ? NH - 1 - w / 2 : w / 2;   // rows down one column, up the next: the A pair stays over the turn
            if constexpr (hs == 0) {
                if constexpr (w == 0) {
                    constexpr int own = 2 * (j < NH ? j : NH);
                    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 2 * (NBN - 1 - j) + own));
                    __builtin_amdgcn_sched_barrier(0);
                }
                // its own reads: two per column in the first NH columns
                if constexpr (j < NH && w < 2) read_a(slot_reads_a, w, NH + j);
            } else if constexpr (NEXT) {
                if constexpr (sl < COL) read_a(slot_reads_a, sl & 1, sl / 2);
                if constexpr (w == 0 && j > 0) {
                    read_b(slot_next_b, 0, j - 1);
                    read_b(slot_next_b, 1, j - 1);
                }
            }
            if constexpr (C2 && sl % CP_EVERY == CP_EVERY / 2)
                issue_one(kt + DEPTH, slot_copy, std::integral_constant<bool, hs == 0>{}, template_int<sl / CP_EVERY>{});
            __builtin_amdgcn_sched_barrier(0);   // nothing moves across an MFMA
            // operands swapped (B rows as the MFMA "A" matrix): a lane ends up with 4 consecutive n for one m
            Mma<T>::run(fb[h][j], fa[h][i0 + r], acc[i0 + r][j]);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (hs == 1 && NEXT) {
            read_b(slot_next_b, 0, NBN - 1);
            read_b(slot_next_b, 1, NBN - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // after: how many panels follow panel kt, DEPTH if at least that many.
    auto kstep = [&](int kt, int sa, int na, int nb, int sp, auto after_c) {
        constexpr int AFTER = decltype(after_c)::value;
        constexpr bool NEXT = AFTER > 0, C2 = AFTER == DEPTH;
        const std::bool_constant<NEXT> next_c;
        const std::bool_constant<C2> c2_c;
        half_step(template_int<0>{}, kt, sa, 0, sp, next_c, c2_c);
        __builtin_amdgcn_sched_barrier(0);
        wait_lds_reads();                 // the A fragments of the second half step; panel kt has been read
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NEXT) {
            // Panel kt+1 has landed for every wave (the copies of the panels behind it and of
            // B(kt+DEPTH), the newest of this wave, may still be in flight: copies complete in
            // issue order), and every wave has read panel kt for the last time.
            wait_vmcnt<C2 ? (DEPTH - 2) * (LOADS_A + LOADS_B) + LOADS_B : (AFTER - 1) * (LOADS_A + LOADS_B)>();
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        half_step(template_int<1>{}, kt, na, nb, sa, next_c, c2_c);
    };

    // Prologue: panels 0 .. DEPTH-1 go out; wait for panel 0.  (Where K has fewer, the last one is
    // copied again, to slots that nobody reads: without branches the waits that the compiler derives
    // for the slot lookups count all of these copies.)
    template_int<0> first_half;
    template_int<1> second_half;
    auto last_panel_next = [&](bool is_last) {   // called before the copies of a panel are issued
        if (is_last) {
            vo0 = tail_off0;
            vo1 = tail_off1;
        }
    };
    static_for<DEPTH>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        const int panel = min(i, NP - 1);
        last_panel_next(panel == NP - 1);
        issue_unit(panel, i * PANEL_A, unit_a, first_half);
        issue_unit(panel, i * PANEL_A, unit_a, second_half);
        issue_unit(panel, B_RING + i * PANEL_B, unit_b, first_half);
        issue_unit(panel, B_RING + i * PANEL_B, unit_b, second_half);
    });
    // The accumulators are cleared here, under the latency of those copies, by MFMAs on zero
    // operands (0 x 0 + 0).  Written as assignments of zero, the compiler places the 256 register
    // writes directly in front of the main loop, behind the wait for the first panel.
    {
        frag zeros;
        asm volatile("v_mov_b32 %0, 0\n\tv_mov_b32 %1, 0\n\tv_mov_b32 %2, 0\n\tv_mov_b32 %3, 0\n\ts_nop 7"
                     : "=v"(((float*)&zeros)[0]), "=v"(((float*)&zeros)[1]), "=v"(((float*)&zeros)[2]),
                       "=v"(((float*)&zeros)[3]));
#pragma unroll
        for (int i = 0; i < NBM; ++i)
#pragma unroll
            for (int j = 0; j < NBN; ++j) Mma<T>::clear(zeros, acc[i][j]);
    }
    if (NP > 1) wait_vmcnt<(DEPTH - 1) * (LOADS_A + LOADS_B)>(); else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    // fragments of the first half step, in the order the main loop leaves them for the next k-step
#pragma unroll
    for (int r = 0; r < 2 * NH; ++r) read_a(0, r & 1, r / 2);
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
        read_b(B_RING, 0, j);
        read_b(B_RING, 1, j);
    }
    __builtin_amdgcn_sched_barrier(0);
    resolve_destination();
    __builtin_amdgcn_sched_barrier(0);

    // The consumer's waves share SIMDs with these waves while a group is being
    // copied; the issue arbiter should always prefer the wave that feeds the MFMAs.
    __builtin_amdgcn_s_setprio(3);
    int kt = 0;
    int ring_a[DEPTH], ring_b[DEPTH + 1];   // the slots, from those of A(kt) and B(kt) on
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) ring_a[u] = u * PANEL_A;
#pragma unroll
    for (int u = 0; u <= DEPTH; ++u) ring_b[u] = B_RING + u * PANEL_B;
    auto rotate = [&]() {
        const int a0 = ring_a[0], b0 = ring_b[0];
#pragma unroll
        for (int u = 0; u + 1 < DEPTH; ++u) ring_a[u] = ring_a[u + 1];
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) ring_b[u] = ring_b[u + 1];
        ring_a[DEPTH - 1] = a0;
        ring_b[DEPTH] = b0;
    };
    if constexpr (MTM == MTN) {
        for (; kt < NP - DEPTH; ++kt) {
            last_panel_next(kt + DEPTH + 1 == NP);   // this k-step copies panel kt + DEPTH
            kstep(kt, ring_a[0], ring_a[1], ring_b[1], ring_b[DEPTH], template_int<DEPTH>{});
            rotate();
        }
    } else {
        // Before one k-step the copies change: they turn back to the first panel, or are those of the last one.  (Never both: where
        // they turn no panel is partial, and the last one's offsets are those of all.)  Asked for in every k-step, by compares and
        // selects, it took 1 % longer with cached operands, 5 % where M or N is ragged (110 shapes).
        int stop = turn ? NP - turn - DEPTH : NP - DEPTH - 1;
        while (kt < NP - DEPTH) {
            if (kt == stop) {
                last_panel_next(true);
                k_first -= turn ? NP : 0;
                stop = NP - DEPTH;
            }
            do {
                kstep(kt, ring_a[0], ring_a[1], ring_b[1], ring_b[DEPTH], template_int<DEPTH>{});
                rotate();
            } while (++kt < stop);
        }
    }
    static_for<DEPTH>([&](auto t_c) {
        constexpr int after = DEPTH - 1 - decltype(t_c)::value;
        if (after == 0 || NP > after) {
            kstep(kt, ring_a[0], ring_a[1], ring_b[1], ring_b[DEPTH], template_int<after>{});
            rotate();
            ++kt;
        }
    });

    // ---- epilogue: registers -> LDS strip -> global -------------------------------
    // acc[i][j][r] is element m = 16i + l%16, n = 16j + 4(l/16) + r (fr_g = l/16).
    __builtin_amdgcn_s_setprio(0);
    settle_mfma();
    __builtin_amdgcn_sched_barrier(0);   // no accumulator read is scheduled ahead of the delay
    if constexpr (MTM == 64) {
        if (part >= 0) {
            // The parts of a 64x64 tile are added up by whichever workgroup finishes last: the others leave their sums
            // with write-through stores, wait for the acknowledgement and count themselves; the last one reads them with
            // loads that are served beyond this XCD's caches, adds in the order of k, its own from registers, and goes on
            // to the epilogue.  Nobody waits for another workgroup.  In 2 to 6 parts this is 16 to 80 KiB to read;
            // a 128x128 tile's 64 KiB a part, at the 43 bytes per ns that one CU gets, took longer than the reduction's launch
            // (128x4096x7168 with its norm: 25.6 us in 4 parts here, 21.7 in 8 with the launch, 20.2 in two of 64x64).
            constexpr int NB = NBM * NBN;
            const __amdgpu_buffer_rsrc_t prsrc = __builtin_amdgcn_make_buffer_rsrc(p.partial, 0, 0xffffffff, 0x00020000);
            const int at = (int)(partial_at(p, tile, 0, wave, NB) * sizeof(f32x4)) + lane * (int)sizeof(f32x4);
            const int next = 4 * NB * 64 * (int)sizeof(f32x4);   // bytes of a part of the tile
            const int inside = live ? valid_m - wm * WM : 0;     // rows of the quadrant inside the matrix
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (16 * (b / NBN) < inside) {
                    f32x4 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = acc_read(acc[b / NBN][b % NBN][r]);
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), prsrc, at + b * 1024, part * next, 16);
                    // (the next reads are assembly the compiler cannot see into: not into the registers of a store just issued)
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_nop 1");
                    __builtin_amdgcn_sched_barrier(0);
                }
            wait_vmcnt<0>();
            __syncthreads();   // also: every wave is done with the panel buffers
            int* before = (int*)smem;
            if (tid == 0) *before = __hip_atomic_fetch_add(p.arrived + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (*before != p.splits - 1) return;
            if (tid == 0) __hip_atomic_store(p.arrived + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next call
            u32x4 other[kMaxHereSplits][NB];
#pragma unroll
            for (int s = 0; s < kMaxHereSplits; ++s)
                if (s < p.splits && s != part)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        if (16 * (b / NBN) < inside) other[s][b] = __builtin_amdgcn_raw_buffer_load_b128(prsrc, at + b * 1024, s * next, 16);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f32x4 own, sum;
#pragma unroll
                for (int r = 0; r < 4; ++r) own[r] = acc_read(acc[b / NBN][b % NBN][r]);
#pragma unroll
                for (int s = 0; s < kMaxHereSplits; ++s)
                    if (s < p.splits) {
                        const f32x4 add = s == part ? own : __builtin_bit_cast(f32x4, other[s][b]);
                        sum = s == 0 ? add : sum + add;
                    }
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[b / NBN][b % NBN][r] = acc_write(sum[r]);
            }
        }
    } else if (part >= 0) {   // a part of a split tile: the sums as they are
        f32x4* out = (f32x4*)p.partial + partial_at(p, tile, part, wave, NBM * NBN) + lane;
#pragma unroll
        for (int b = 0; b < NBM * NBN; b += 4)
            if (live && 16 * (b / NBN) < valid_m - wm * WM) {   // not the blocks below the matrix
                f32x4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[k][r] = acc_read(acc[(b + k) / NBN][(b + k) % NBN][r]);
#pragma unroll
                for (int k = 0; k < 4; ++k) out[(b + k) * 64] = v[k];
                // (the next reads are assembly the compiler cannot see into: not into the registers of a store just issued)
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_nop 1");
                __builtin_amdgcn_sched_barrier(0);
            }
        return;
    }
    __syncthreads();  // every wave is done with the panel buffers
    if constexpr (MODE == kScatter)
        if (deliver) {
            dl_lo = receive_row(p, re_lo, tile_group);
            if constexpr (WM > 64) dl_hi = receive_row(p, re_hi, tile_group);
        }
    constexpr int PITCH = WN * 2 + 16;                  // strip row pitch in bytes
    constexpr int ROWCH = WN / 8;                       // 16-byte chunks per strip row
    // Two strip buffers per wave, used in turn: the next strip is written while this one is being stored.
    unsigned char* ep0 = smem + wave * (32 * PITCH);
    unsigned char* ep1 = ep0 + 4 * 32 * PITCH;
    T* D = (T*)p.D;
    T* D2 = (T*)p.D2;
    [[maybe_unused]] __amdgpu_buffer_rsrc_t drsrc, d2rsrc;
    if constexpr (STORE == 1) drsrc = __builtin_amdgcn_make_buffer_rsrc(p.D, 0, 0xffffffff, 0x00020000);
    if constexpr (MODE != kScatter) d2rsrc = __builtin_amdgcn_make_buffer_rsrc(p.D2, 0, 0xffffffff, 0x00020000);
    // Cache policies of the buffer stores (the aux operand on gfx950).
    [[maybe_unused]] constexpr int kNonTemporal = 2, kWriteThrough = 16;
    // D of a call that delivers every tile: nobody polls for it and its copy is what is read next.
    [[maybe_unused]] const bool stream_c = p.D2 && (MODE == kPlain || p.deliver_from == 0);
#pragma unroll
    for (int i = 0; i < NBM / 2; ++i) {   // strip i: rows 32i .. 32i+31 of the quadrant
        unsigned char* ep = (i & 1) ? ep1 : ep0;
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
            for (int j = 0; j < NBN; ++j) {
                out4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = (T)acc_read(acc[2 * i + ii][j][r]);
                *(out4*)(ep + (16 * ii + fr_row) * PITCH + (16 * j + 4 * fr_g) * 2) = o;
            }
#pragma unroll
        for (int it = 0; it < WN / 16; ++it) {
            const int c = it * 64 + lane;
            const int r = c / ROWCH, cc = c % ROWCH;
            const u32x4 v = *(const u32x4*)(ep + r * PITCH + cc * 16);
            int row = row0 + 32 * i + r;
            if constexpr (MODE == kScatter) {
                const int q_row = 32 * i + r;   // row within the quadrant: held by lane q_row % 64
                row = __shfl((WM > 64 && i >= 2) ? re_hi : re_lo, q_row & 63, 64);
                if (deliver) {
                    const int recv = __shfl((WM > 64 && i >= 2) ? dl_hi : dl_lo, q_row & 63, 64);
                    if (live && recv >= 0) *(u32x4*)(D2 + (size_t)recv * ld + col0 + cc * 8) = v;
                }
            }
            const size_t off = (size_t)row * ld + col0 + cc * 8;
            if (!live) continue;   // a quadrant outside the matrix goes through the motions and stores nothing
            if constexpr (EDGE) {
                const int gcol = col0 + cc * 8;
                if (row >= p.M || gcol >= p.N) continue;
                if (p.ld & 7) {    // rows of D are not 16-byte aligned
                    store_edge_chunk(D + off, v, p.N - gcol);
                    if (deliver) store_edge_chunk(D2 + off, v, p.N - gcol);
                    continue;
                }
            }
            if (MODE != kPlain && !D) {
                // (delivered only)
            } else if constexpr (STORE == 1) {
                if (stream_c) __builtin_amdgcn_raw_buffer_store_b128(v, drsrc, (int)(off * 2), 0, kNonTemporal);
                else __builtin_amdgcn_raw_buffer_store_b128(v, drsrc, (int)(off * 2), 0, kWriteThrough);
            } else {
                *(u32x4*)(D + off) = v;
            }
            if constexpr (MODE != kScatter)
                if (deliver) {
                    if (p.stream_deliver) __builtin_amdgcn_raw_buffer_store_b128(v, d2rsrc, (int)(off * 2), 0, kNonTemporal);
                    else __builtin_amdgcn_raw_buffer_store_b128(v, d2rsrc, (int)(off * 2), 0, 0);
                }
        }
    }

    // ---- signal ---------------------------------------------------------------------
    if constexpr (MODE != kPlain) {
        if (p.D2 && p.deliver_from == 0) return;   // nothing is signalled
        // Every wave's tile stores are acknowledged before the barrier: with
        // write-through stores they are then visible device-wide (REL = 1);
        // otherwise the release on the atomic writes this L2's dirty lines back
        // before the counter moves.
        wait_vmcnt<0>();
        __syncthreads();
        const int ntile = (MTM >> p.log_bm) * (MTN >> p.log_bn);
        // The tiles of a macro tile mostly fall into one group: the first lane of
        // every distinct group adds that group's tile count in one atomic (at most
        // four lanes take part, all in the first wavefront).  Monitor mode keeps
        // one atomic per tile, like the reference: the tickets are per tile.
        int same = 0, earlier = 0;
        if (wave == 0) {
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                const int g = __shfl(sig_group, o, 64);
                if (o < ntile && g == sig_group && g >= 0) {
                    ++same;
                    if (o < tid) ++earlier;
                }
            }
        }
        if (tid < ntile && sig_group >= 0 && (p.monitor || earlier == 0)) {
            const int add = p.monitor ? 1 : same;
            if constexpr (REL == 1)  // the stores already went through to memory
                __hip_atomic_fetch_add(p.MM + sig_group, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else
                __hip_atomic_fetch_add(p.MM + sig_group, add, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            if (p.monitor) {
                const int order =
                    __hip_atomic_fetch_add(p.MM + p.TN - 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                p.MM[p.TN + sig_slot] = order;
            }
        }
    }
}


// SMEM: the panel slots (160 KiB at MTM = 256).
template <auto KERN, int SMEM>
static int launch_gemm_kernel(const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    // The attribute belongs to the function on one device: set it once per device.
    static std::atomic<unsigned long long> configured{0};
    int dev = 0;
    FO_HIP(hipGetDevice(&dev));
    const unsigned long long bit = 1ull << (dev & 63);
    if (!(configured.load(std::memory_order_acquire) & bit)) {
        FO_HIP(hipFuncSetAttribute((const void*)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM));
        configured.fetch_or(bit, std::memory_order_release);
    }
    const int grid = p.split_from + p.split_tiles * p.splits;
    if (timer.start || timer.stop) hipExtLaunchKernelGGL(KERN, dim3(grid), dim3(256), SMEM, stream, timer.start, timer.stop, 0, p);
    else hipLaunchKernelGGL(KERN, dim3(grid), dim3(256), SMEM, stream, p);
    FO_HIP(hipGetLastError());
    return FO_OK;
}

}  // namespace fo
