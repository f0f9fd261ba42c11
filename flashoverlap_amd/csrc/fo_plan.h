// Which macro tile computes a shape, and which tiles are split over K: the estimate and the choice, on the host alone.
#pragma once

#include <algorithm>
#include <cstddef>

#include "../../include/flashoverlap_hip.h"
#include "fo_raster.h"

namespace fo {

constexpr int kBK = 64;             // k-elements per LDS buffer
constexpr int kMaxHereSplits = 6;   // parts of a 64x64 tile, added up in the GEMM
constexpr int kTurnFrom = 48;       // panels of K from which on the XCDs begin at different ones (turn_panels)
constexpr int kLowRow = 200;        // rows of the matrix, at most, in a last row of 256x128 tiles that is low
constexpr int kThinColumn = 32;     // columns of it in a last column of tiles whose workgroups run ahead
constexpr size_t kMaxWorkspace = (size_t)64 << 20;   // bytes of the parts of split tiles, at most
constexpr int kSkinnyRows = 32;     // rows that the skinny kernel takes (fo_internal.h has its times)

struct Macro {
    int m, n;
};

// How a shape is computed: the macro tile, and which macro tiles are split over K.
struct Plan {
    Macro macro;
    int from, tiles, splits, panels;   // the last `tiles` macro tiles, in `splits` parts of `panels` panels; 0: none
    size_t bytes;                      // workspace of the parts
    double us;                         // estimated
    int strip_m, strip_n;              // the last rows or columns of D that a skinny GEMM computes (at most one of the two)
};

// Estimated microseconds of a GEMM in macro tiles of one kind.  Fitted on 1138 shapes of 33 to 16384 rows, 512 to 8192
// columns and K 512 to 8192, fp16 and bf16, each timed in the tiles and splits that come near (some 6000 kernels), with operands
// from HBM and with operands that the memory-side cache holds, so that the plans taken are short in both and few are much longer
// than the fastest one measured.  On 334 other shapes the plan taken is on average 1.3 % (HBM) and 0.9 % (cached) slower than
// the fastest, 23 and 17 % at worst; with the constants before, which were fitted to the times, 1.6 and 0.8 %, 37 and 17 % at
// worst.  Those priced parts of 256x256 tiles too low, and lone 128x128 tiles with operands from HBM.  us, HBM and cached, before | now:
// 2041x4096x7168 fp16 113.0 111.2 | 104.2 101.5, 77x7680x7936 bf16 33.9 25.7 | 29.8 25.0, 4608x1152x4544 fp16 68.2 53.6 | 61.6 50.0,
// 6683x1336x1600 bf16 51.6 38.9 | 38.6 37.0, 640x3840x7872 fp16 74.4 51.0 | 52.1 52.4.
// With more than half of the CUs at work all the time the k-steps of the larger tiles get longer; at the chip's power limit, in
// several full rounds, by more than is said here, but no other tile comes near 256x256 there.
// (256x128 tiles are priced as they were before K was begun apart in them and their loop lost its selects: they are now up to a tenth
// shorter.  Of 70 shapes given to other tiles by less than 12 %, 30 would be 3 to 14 % faster in them; over all 70 the choice is level.)
struct Shape {
    int panels, cus;
    double straddle;     // rows that do not start on cache lines ask the L2 for a line twice: all of them, or half where K is a multiple of 32
    double operands_us;  // A and B at 8.4 TB/s
    double out_mb;       // D, in 10^6 bytes
};
// 64x64 in `parts` parts each.  One to a CU, or two, each of which then hides the other's latency.  The parts are added up
// by the workgroup that finishes last, the more of them the longer (fo_gemm_body.h).
inline double us_64(const Shape& s, int total, int parts, int per) {
    const double load = (double)total * parts / s.cus;
    const double step = load <= 1.0 ? 0.172 + ((parts == 1 ? 0.035 : 0.0) + 0.06 * load) * s.straddle + 0.023 * load : 0.375 + 0.165 * s.straddle;
    return 2.9 + std::max(per * step, s.operands_us) + (parts > 1 ? 2.0 + 0.35 * parts : 0.0);
}
// 128x128, `rest` of them in `parts` parts behind `whole` times as many whole tiles as CUs.  While they fit one to a CU they
// have the ring of four panels; of more than that a CU holds two, and while one starts or stores the other multiplies: they take
// k-steps only.  That also pairs them up as they come: parts behind an odd number of whole tiles to a CU share
// theirs with a whole one, behind an even number with each other.  Where few tiles are left over, the CUs that hold two have more of the
// L2 to themselves, but with rows off the cache lines that is little of a relief (2176x2304x632, 306 tiles: 15.9 us, 13.5 in 256x128
// ones with operands that are cached).  The parts are written and read again, by a second launch.
inline double us_128(const Shape& s, int whole, int rest, int parts, int per) {
    const double load = (double)rest * parts / s.cus, add = parts > 1 ? 0.86 + 0.023 * rest * parts : 0.0;
    if (whole == 0) return 4.06 + std::max(per * (0.458 + 0.155 * s.straddle), s.operands_us) + add;
    const double alone = parts > 1 ? (whole % 2 ? 1.0 : 0.5) : 0.5 + 0.4 * s.straddle, last = alone + (1.0 - alone) * load;
    return 2.12 + (0.497 + 0.168 * s.straddle) * (s.panels * whole + per * last) + add + 0.144 * s.out_mb;
}
// The larger tiles have a CU to themselves, and a round of them takes as long if it is not full.
inline double hot(double busy) { return std::min(1.0, std::max(0.0, 2.0 * busy - 1.0)); }
inline double us_256(const Shape& s, int whole, int rest, int parts, int per) {
    auto round_us = [&](double busy, int panels) { return 8.63 + panels * (1.107 + 0.145 * hot(busy) + 0.087 * s.straddle * (1.0 - hot(busy))); };
    const double load = (double)rest * parts / s.cus;
    if (parts > 1) return whole * round_us(1.0, s.panels) + round_us(load, per) + 0.072 * rest * parts;
    return (whole + 1) * round_us((whole + load) / (whole + 1), s.panels);
}
inline double us_256x128(const Shape& s, int whole, int rest) {
    const double busy = (whole + (double)rest / s.cus) / (whole + 1);
    return (whole + 1) * (4.98 + s.panels * (0.662 + std::max(0.043 * hot(busy), 0.219 * s.straddle))) + 0.125 * s.out_mb;
}

// The plan whose estimated time is the smallest.  Of a round that is at most half full the 128x128 and 256x256 tiles can be
// split over K; 64x64 tiles are all split or none, while they come to two workgroups a CU at most.
inline Plan make_plan(int BM, int BN, int M, int N, int K, bool any_tile, bool may_split, bool all_tiles, Macro forced, int cus) {
    const Shape s{(K + kBK - 1) / kBK, cus, K % kBK == 0 ? 0.0 : K % 32 == 0 ? 0.5 : 1.0, ((double)M + N) * K * 2 / 8.4e6, (double)M * N * 2e-6};
    Plan best{};
    double best_us = 1e30;
    for (const Macro t : {Macro{256, 256}, Macro{256, 128}, Macro{128, 128}, Macro{64, 64}}) {
        if (forced.m ? t.m != forced.m || t.n != forced.n : !any_tile && (t.m % BM || t.n % BN)) continue;
        if ((t.m != t.n || t.m == 64) && !all_tiles) continue;
        const int total = ((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n);
        if (t.m == 64 && total > 2 * cus) continue;
        const int whole = t.m == 64 ? 0 : (total - 1) / cus, rest = total - whole * cus;
        const int most = !may_split || t.m != t.n ? 1 : t.m == 64 ? kMaxHereSplits : t.m == 128 ? 10 : 16;
        for (int n = 1; n <= most; ++n) {
            const int per = (s.panels + n - 1) / n, parts = (s.panels + per - 1) / per;
            if (n > 1 && (per < (t.m == 64 ? 3 : 4) || rest * n > (t.m == 64 ? 2 * cus : cus))) break;
            if (parts != n) continue;   // (the same as with fewer)
            const size_t bytes = n == 1 ? 0 : FO_WORKSPACE_ZEROED + (size_t)rest * n * t.m * t.n * sizeof(float);
            if (bytes > FO_WORKSPACE_ZEROED + kMaxWorkspace) break;
            const double us = t.m == 64 ? us_64(s, total, n, per) : t.m == 128 ? us_128(s, whole, rest, n, per)
                              : t.n == 256 ? us_256(s, whole, rest, n, per) : us_256x128(s, whole, rest);
            if (us >= best_us) continue;
            best_us = us;
            best = n == 1 ? Plan{t, total, 0, 1, s.panels, 0, us} : Plan{t, total - rest, rest, n, per, bytes, us};
        }
    }
    return best;
}

// 256x128 tiles in one round: the panels of K between the places at which the XCDs begin (fo_gemm_body.h), 0 if all begin at the first.
// Workgroups in step ask for the same few columns of every row at a time; apart, an XCD finds what another one has read already in the
// memory-side cache.  So it pays where the XCDs share the rows of A: where every band of four rows of tiles, the last one too, has at
// least a column of its tiles on a second XCD.  Rows that one XCD has to itself come from HBM all the same, now while the others do not wait for
// the same columns, and that is slower, unless the last row of tiles is low.  Where the last column of tiles has few columns of the matrix its
// workgroups copy less and run ahead by themselves.  (That much is measured; that it is the channels and caches is a conjecture.)
// Operands from HBM, bf16 and fp16, all at panel 0 / apart: 790 shapes of this rule 1.077 (geometric mean; the slowest 0.96), the 466
// others 0.990 (0.93 at worst).  us, K = 4160 bf16: 2048x3328 57.7 / 52.4, 2176x2304 56.9 / 51.0, 3072x2176 58.1 / 53.7; 2304x2304 57.6 / 60.6, 3328x2048
// 58.3 / 61.8, 7168x896 59.7 / 63.5; K = 6272: 2248x3072 87.2 / 81.5, 2280x3072 86.4 / 89.0; 1024x5888 83.8 / 78.5, 1024x5840 82.3 / 80.1,
// 1024x5792 77.3 / 79.5.  From the memory-side cache level (110 shapes 0.9995, 0.991 at worst).  From 48 panels on: the gain begins earlier
// (2048x4096x2432 39.8 / 38.8, 640x8832x2048 30.2 / 29.0), but was measured on six shapes there, not on this range.
inline int turn_panels(Macro macro, int M, int N, int K, int cus) {
    if (macro.m == macro.n || K % kBK || K / kBK < kTurnFrom) return 0;
    constexpr int kBand = kGroupM / 2;
    const int GM = (M + macro.m - 1) / macro.m, GN = (N + macro.n - 1) / macro.n, tiles = GM * GN;
    const int last_band = (GM - 1) % kBand + 1, last_row = M - (GM - 1) * macro.m, last_column = N - (GN - 1) * macro.n;
    if (tiles > cus || last_column <= kThinColumn) return 0;
    // a band of that many rows exceeds an XCD's share of the tiles, by at least so many
    auto exceeds = [&](int rows, int by) { return (rows * GN - by) * kXcds >= tiles; };
    if (GM > kBand && !exceeds(kBand, kBand)) return 0;
    const bool low = last_row <= kLowRow && (last_band == 1 || exceeds(last_band, 1));
    return low || exceeds(last_band, last_band) ? K / kBK / kXcds : 0;
}

// A plain GEMM of which a few rows or columns lie behind the last whole multiple of 128: as macro tiles they are a row or column
// of tiles that multiplies zeros, often a round of its own.  The skinny kernel (with the operands exchanged, for columns) reads the
// other operand once more, at HBM's rate if it is large, and starts like any launch.  It runs in front of the tiles, which then
// find that operand in the memory-side cache.  Taken where that is estimated to be shorter by 5 %, or by 8 us (the rounds that both have
// in common err alike), and where the rows of the operands start on cache lines: the estimates of others err by up to a third, which
// only columns, whose tiles also store ragged rows, make up for.  On 80 shapes for which it is estimated to be so, time / time in
// tiles: strips of columns 0.92 (1.01 at worst), with K an odd multiple of 32 0.88 (1.02), of rows 0.96 (1.02) and 0.99 (1.24, not taken).
// Plain GEMM, its bulk copy and the norm, us, in tiles / so: 8191x4097x7168 bf16 353 / 339, 8192x4104x1024 106 / 93,
// 2080x4112x4096 fp16 85 / 78.
inline double us_strip(int other_rows, int K) { return 4.5 + (double)other_rows * K * 2 / 5.2e6; }
inline void consider_strip(Plan* plan, int BM, int BN, int M, int N, int K, bool may_split, bool all_tiles, int cus) {
    const int rest_m = M % 128, rest_n = N % 128;
    auto consider = [&](int sm, int sn) {
        const double strip = us_strip(sm ? N : M, K);
        if (M - sm <= 0 || N - sn <= 0 || strip >= plan->us) return;
        Plan other = make_plan(BM, BN, M - sm, N - sn, K, true, may_split, all_tiles, Macro{0, 0}, cus);
        if (!other.macro.m || other.us + strip >= plan->us - std::min(0.05 * plan->us, 8.0)) return;
        *plan = other;
        plan->us = other.us + strip;
        plan->strip_m = sm;
        plan->strip_n = sn;
    };
    if (rest_m && rest_m <= kSkinnyRows && K % 64 == 0) consider(rest_m, 0);
    if (rest_n && rest_n <= kSkinnyRows && K % 32 == 0) consider(0, rest_n);
}

}  // namespace fo
