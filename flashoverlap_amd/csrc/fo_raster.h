// Workgroup -> macro-tile rasterisation, shared by the GEMM kernels (device)
// and fo_raster_hint (host) so that both sides agree on the issue order.
//
// MI355X dispatches workgroup i of a grid to XCD i % 8, and every XCD has its
// own L2.  The unit of the map is a block of kGroupM x 4 macro tiles: the 32
// workgroups one XCD runs at a time, which share their A and B panels in that
// L2 (numbered row by row inside the block).  Units are ordered band by band (a band = kGroupM rows of macro tiles,
// all columns), and the eight units of one hardware wave (256 workgroups) go to
// the eight XCDs.  So the XCDs of a wave work on the same A rows, which the
// memory-side cache then fetches from HBM once for all of them (with each XCD
// walking a strip of its own the same kernel ran 2 % longer on operands that
// were not cached), and a wave finishes whole rows of the output.
#pragma once

#if defined(__HIPCC__)
#define FO_HD __host__ __device__ inline
#else
#define FO_HD inline
#endif

namespace fo {

constexpr int kXcds = 8;
constexpr int kGroupM = 8;   // rows of a unit
constexpr int kUnitN = 4;    // columns of a unit: kGroupM * kUnitN = 32 workgroups, one XCD's share of a wave

struct TileCoord {
    int m, n;
};

// Division by the column count without a divide instruction (the kernel does this once per
// workgroup, in front of its first memory access): n / d == (n * magic) >> 32 with
// magic = 2^32 / d + 1, exact while n * d < 2^32 (tile counts are far below that).
// (d = 1 has no such 32-bit magic; it is stored as 0.)
FO_HD unsigned raster_magic(int d) { return d == 1 ? 0u : (unsigned)(0x100000000ull / (unsigned)d) + 1u; }
FO_HD int raster_div(int n, unsigned magic) {
    return magic ? (int)(((unsigned long long)(unsigned)n * magic) >> 32) : n;
}

constexpr int kWave = kXcds * kGroupM * kUnitN;

// n / d for n < 32 and 1 <= d <= 8: n * ceil(256 / d) / 256, the factors less one in the bytes of a constant
// (256 / d is exceeded by at most 7 / d, which 31 * 7 < 256 keeps from reaching the next quotient).
FO_HD unsigned raster_div_small(unsigned n, unsigned d) {
    const unsigned factor = (unsigned)(0x1f242a333f557fffull >> (8 * (d - 1))) & 255;
    return (n * factor + n) >> 8;
}

// Position in unit order -> macro tile coordinate; gn_magic = raster_magic(GN).  kGroupM x kUnitN: the
// unit, 8 x 4 square macro tiles, 4 x 8 of those that are twice as high as wide.  Blocks that begin at
// position by_column or later are numbered column by column.
template <int kGroupM = fo::kGroupM, int kUnitN = fo::kUnitN>
FO_HD TileCoord raster_tile(int pos, int GM, int GN, unsigned gn_magic, int by_column) {
    static_assert(kGroupM * kUnitN * kXcds == kWave, "a unit is an XCD's share of a wave");
    // Position -> tile: bands of kGroupM rows (the last may be lower), in a band blocks of kUnitN
    // columns (the last may be narrower), in a block row by row.  (Row by row, not column by
    // column: the slots of the tiles that one output row crosses are then a few slots apart
    // inside a block and one block apart between blocks, where column by column they were 256
    // slots = 8 MiB apart, a stride at which the segments that reorder+RMSNorm gathers for a row
    // fall into few memory channels: that kernel ran 5-7 % longer.)
    // (Unsigned, with one divide and that only in a band that is not whole, and next to no branches: all of this
    // stands in front of a workgroup's first memory access.)
    const unsigned at = (unsigned)pos;
    const unsigned first_m = (unsigned)raster_div((int)(at / kGroupM), gn_magic) * kGroupM;   // at / (kGroupM * GN)
    const unsigned in_band = at - first_m * (unsigned)GN;
    const unsigned rows = (unsigned)GM - first_m >= kGroupM ? kGroupM : (unsigned)GM - first_m;
    unsigned block = in_band / (kGroupM * kUnitN);   // (the band's last one can be narrower)
    if (__builtin_expect(rows != kGroupM, 0)) block = in_band / (rows * kUnitN);
    const unsigned in_block = in_band - block * rows * kUnitN, first_n = block * kUnitN;
    const unsigned cols = (unsigned)GN - first_n >= kUnitN ? kUnitN : (unsigned)GN - first_n;
    const bool columns = at - in_block >= (unsigned)by_column;
    const unsigned run = columns ? rows : cols;
    const unsigned major = raster_div_small(in_block, run), minor = in_block - major * run;
    const unsigned r = columns ? minor : major, col = columns ? major : minor;
    return {(int)(first_m + r), (int)(first_n + col)};
}

FO_HD int raster_whole(int total) { return (int)((unsigned)total / kWave * kWave); }   // workgroups in whole waves

// Workgroup pid in [0, total) -> position: workgroup `local` of XCD `xcd` is workgroup local % 32 of that
// XCD's unit in wave local / 32.  The workgroups behind the last whole wave are shared out in the same way, in
// eight runs of positions, there column by column (by_column = raster_whole): a run then crosses all rows of its band and as few
// columns as can be, wherever it begins.  (With a position equal to the workgroup's number every XCD took
// every eighth tile: plain 7168x1152x3520 bf16 64.5 us in 252 tiles of 256x128,
// 50.9 like this; 7168x1152x3512 76.0 and 71.9; 4381x1144x4672 53.8 and 49.2.  Row by row the runs cross two blocks and
// twice the columns: 992x6496x4232, four rows of tiles, 68.3, 79.8 and by column 68.6.)
FO_HD int raster_pos(int pid, int total) {
    constexpr unsigned kUnit = kGroupM * kUnitN;
    const unsigned xcd = (unsigned)pid % kXcds, local = (unsigned)pid / kXcds;
    const unsigned whole = (unsigned)raster_whole(total), rest = (unsigned)total - whole;
    const unsigned per = rest / kXcds, more = rest % kXcds;   // the first `more` XCDs have one more
    const unsigned in_wave = (local / kUnit * kXcds + xcd) * kUnit + local % kUnit;
    const unsigned behind = whole + xcd * per + (xcd < more ? xcd : more) + (local - whole / kXcds);
    return (int)((unsigned)pid < whole ? in_wave : behind);
}

template <int kGroupM = fo::kGroupM, int kUnitN = fo::kUnitN>
FO_HD TileCoord raster_map(int pid, int GM, int GN, unsigned gn_magic) {
    return raster_tile<kGroupM, kUnitN>(raster_pos(pid, GM * GN), GM, GN, gn_magic, raster_whole(GM * GN));
}

// The order that fo_raster_hint reports.  Workgroups of a wave finish together, so behind the last whole wave
// it is free, and goes by position, row by row: for the kernel that gathers output rows (see raster_tile).
template <int kGroupM = fo::kGroupM, int kUnitN = fo::kUnitN>
FO_HD TileCoord raster_order(int pid, int GM, int GN, unsigned gn_magic) {
    const int total = GM * GN;
    return raster_tile<kGroupM, kUnitN>(pid < raster_whole(total) ? raster_pos(pid, total) : pid, GM, GN, gn_magic, total);
}

}  // namespace fo
