// The square macro tiles of the GEMM (its kernel body is fo_gemm_body.h) and what every GEMM call goes
// through: validation, the choice of the macro tile and of the tiles to split over K, the launch.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <string_view>
#include <type_traits>
#include <utility>

#include "fo_gemm_body.h"
#include "fo_internal.h"
#include "fo_knobs.h"
#include "fo_plan.h"
#include "fo_raster.h"

namespace fo {

template <typename T, int MT, int MODE, int STORE, int REL, bool EDGE = false>
__global__ void __launch_bounds__(256) gemm_kernel(const GemmParams p) {
    gemm_body<T, MT, MT, MODE, STORE, REL, EDGE>(p);
}

template <typename T, int MT, int MODE, int STORE, int REL, bool EDGE = false>
static int launch_one(const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    return launch_gemm_kernel<gemm_kernel<T, MT, MODE, STORE, REL, EDGE>, ring_bytes(MT, MT, 2)>(p, timer, stream);
}

template <typename T, int MT>
static int launch_mt(int mode, bool edge, const GemmParams& p, const LaunchTimer& timer, hipStream_t stream) {
    // fo_tune knobs (how the epilogue stores C and how it signals), each read once per launch
    const int store_mode = knob(knobs().store_mode), release_mode = knob(knobs().release_mode);
    const int store = mode == kPlain ? (store_mode ? 1 : 0) : (store_mode || release_mode ? 1 : 0);
    const int rel = (mode != kPlain && release_mode) ? 1 : 0;
    if (mode == kPlain && edge)
        return store ? launch_one<T, MT, kPlain, 1, 0, true>(p, timer, stream) : launch_one<T, MT, kPlain, 0, 0, true>(p, timer, stream);
    if (mode == kPlain)
        return store ? launch_one<T, MT, kPlain, 1, 0>(p, timer, stream) : launch_one<T, MT, kPlain, 0, 0>(p, timer, stream);
    if (mode == kSignal) {
        if (rel) return launch_one<T, MT, kSignal, 1, 1>(p, timer, stream);
        return store ? launch_one<T, MT, kSignal, 1, 0>(p, timer, stream) : launch_one<T, MT, kSignal, 0, 0>(p, timer, stream);
    }
    if (rel) return launch_one<T, MT, kScatter, 1, 1>(p, timer, stream);
    return store ? launch_one<T, MT, kScatter, 1, 0>(p, timer, stream) : launch_one<T, MT, kScatter, 0, 0>(p, timer, stream);
}

static Macro forced_macro(bool any_shape, int BM, int BN) {   // fo_tune; {0, 0}: none that this layout tile allows
    const int f = knob(knobs().macro_tile);
    const Macro t = f == 256128 ? Macro{256, 128} : Macro{f, f};
    return f && (any_shape || (t.m % BM == 0 && t.n % BN == 0)) ? t : Macro{0, 0};
}

// The square macro tile whose issue order fo_raster_hint reports.  Every layout tile (128 or 256 on a
// side) divides 256x256; a matrix edge that is an odd multiple of 128 is covered by half a macro
// tile.  Outputs of up to 128 tiles of 256x256 are one round of smaller tiles, in which the order
// says little about which tile finishes first.
static Macro hint_macro(int BM, int BN, int M, int N) {
    if (const Macro f = forced_macro(false, BM, BN); f.m) return f;
    const int wg256 = ((M + 255) / 256) * ((N + 255) / 256);
    return BM == 128 && BN == 128 && wg256 <= 128 ? Macro{128, 128} : Macro{256, 256};
}

// The store and signal forms of the default: the only ones that all macro tiles are built for.
static bool default_forms() { return knob(knobs().store_mode) && knob(knobs().release_mode); }

static int plan_for(const fo_gemm_call& c, bool workspace, int cus, Plan* plan) {
    int BM, BN, BK;
    if (algo_tile(c.algo, &BM, &BN, &BK) != FO_OK) return fail(FO_ERR_ARG, "fo_gemm: Algo %d out of range", c.algo);
    // Tiles that are signalled take a macro tile of whole layout tiles, tickets are taken in the GEMM's own
    // epilogue, and the signal and store forms behind knobs are built for the two square tiles.
    const bool plain = c.mode == kPlain, any_tile = plain || (c.deliver && c.deliver_from == 0);
    const Macro forced = forced_macro(any_tile, BM, BN);
    *plan = make_plan(BM, BN, c.M, c.N, c.K, any_tile, workspace && (plain || !c.monitor), default_forms(), forced, cus);
    if (!plan->macro.m) *plan = make_plan(BM, BN, c.M, c.N, c.K, any_tile, false, true, forced, cus);
    if (plain && !knob(knobs().macro_tile)) consider_strip(plan, BM, BN, c.M, c.N, c.K, workspace, default_forms(), cus);
    return FO_OK;
}

// A few rows of A: a kernel of its own, unless a macro tile is asked for.
static bool is_skinny(const fo_gemm_call& c) { return c.mode == kPlain && c.M <= kSkinnyRows && !knob(knobs().macro_tile); }

// Sizes with which the kernels' offsets, and make_plan's tile counts, stay inside their types.
static int check_limits(int M, int N, int K) {
    if ((long long)M * N >= (1LL << 31)) return fail(FO_ERR_LIMIT, "fo_gemm: M*N=%lld needs 64-bit tile offsets", (long long)M * N);
    // (the rows a macro tile may reach beyond an operand must still have 32-bit byte offsets)
    if (((long long)M + 256) * K >= (1LL << 31) || ((long long)N + 256) * K >= (1LL << 31))
        return fail(FO_ERR_LIMIT, "fo_gemm: an operand of %lld elements exceeds the 4 GiB a buffer descriptor addresses",
                    (long long)(M > N ? M : N) * K);
    return FO_OK;
}

int gemm_workspace(const fo_gemm_call& c, size_t* bytes) {
    *bytes = 0;
    if (c.M <= 0 || c.N <= 0 || c.K <= 0) return fail(FO_ERR_SHAPE, "fo_gemm_workspace: empty problem %dx%dx%d", c.M, c.N, c.K);
    if (int e = check_limits(c.M, c.N, c.K)) return e;
    if (is_skinny(c)) return FO_OK;
    const DeviceFacts* facts;
    if (int e = device_facts(&facts)) return e;
    Plan plan;
    if (int e = plan_for(c, true, facts->cus, &plan)) return e;
    *bytes = plan.bytes;
    return FO_OK;
}

// A delivered buffer of this many bytes is stored past the memory-side cache, of whose 256 MiB the norm that
// reads it next would find little; a smaller one is left there.  Plain call with its norm, us, left there / past it:
// 8192x4096x1024, 64 MiB, 98 / 103; 12288x8192x1024, 192 MiB, 240 / 253; 16384x7168x1024, 224 MiB, 295 / 289; 16384x8192x1024 and
// x512, 256 MiB, 347 / 323 and 260 / 246; 16384x9216x1024, 288 MiB, 403 / 366; 16384x12288x1024, 384 MiB, 528 / 492;
// 16384x16384x1024 and x512, 512 MiB, 726 / 709 and 576 / 553.
static constexpr long long kStreamDeliverFrom = 256ll << 20;

int launch_gemm(const fo_gemm_call& c, hipStream_t stream, bool keep_d, fo_workspace_fn ask, void* context) {
    const int mode = c.mode, dtype = c.dtype, algo = c.algo, M = c.M, N = c.N, K = c.K, rLDN = c.rLDN, G = c.G;
    const void *A = c.A, *B = c.B;
    void* D = c.D;
    // An event pair armed by fo_time_next_launch belongs to this call whether or not it gets as far
    // as a launch: taken here, ahead of the validation, so that a rejected call cannot leave it
    // behind for some later, unrelated launch.
    LaunchTimer timer = t_launch_timer;
    t_launch_timer = LaunchTimer{};
    if (timer.start) {   // a dispatch that carries events cannot be recorded into a graph
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        FO_HIP(hipStreamIsCapturing(stream, &status));
        if (status != hipStreamCaptureStatusNone)
            return fail(FO_ERR_ARG, "fo_gemm: the event pair of fo_time_next_launch cannot be attached while the stream is being captured");
    }
    int BM, BN, BK;
    if (algo_tile(algo, &BM, &BN, &BK) != FO_OK) return fail(FO_ERR_ARG, "fo_gemm: Algo %d out of range", algo);
    if ((BM != 128 && BM != 256) || (BN != 128 && BN != 256))
        return fail(FO_ERR_ARG, "fo_gemm: layout tile %dx%d: the kernel takes edges of 128 or 256", BM, BN);
    if (dtype != FO_F16 && dtype != FO_BF16) return fail(FO_ERR_ARG, "fo_gemm: dtype %d not fp16/bf16", dtype);
    if (!keep_d) {
        if (mode == kPlain || !c.deliver || c.deliver_from != 0) return fail(FO_ERR_ARG, "fo_gemm_deliver: every tile of a signalling or scattering call has to be delivered");
        D = c.deliver;   // for the checks below
    }
    if (!A || !B || !D) return fail(FO_ERR_ARG, "fo_gemm: null operand");
    if (M <= 0 || N <= 0 || K <= 0) return fail(FO_ERR_SHAPE, "fo_gemm: empty problem %dx%dx%d", M, N, K);
    // The plain GEMM writes a natural row-major D and takes any M and N; the signalling modes place
    // whole layout tiles.
    const bool any_shape = mode == kPlain;
    if (!any_shape && (M % BM || N % BN))
        return fail(FO_ERR_SHAPE, "fo_gemm_signal: M=%d N=%d not multiples of the %dx%d tile", M, N, BM, BN);
    if (K % 8) return fail(FO_ERR_SHAPE, "fo_gemm: K=%d not a multiple of 8 (operand rows must be 16-byte aligned)", K);
    if (int e = check_limits(M, N, K)) return e;
    if (K % kBK && ((long long)M * K >= (1LL << 30) || (long long)N * K >= (1LL << 30)))
        return fail(FO_ERR_LIMIT, "fo_gemm: K=%d is not a multiple of %d and an operand exceeds the 2 GiB this case addresses", K, kBK);
    if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)D) & 15) return fail(FO_ERR_ARG, "fo_gemm: operands must be 16-byte aligned");
    GemmParams p{};
    p.A = A; p.B = B; p.D = D;
    p.M = M; p.N = N; p.K = K; p.ld = N;
    p.BM = BM; p.BN = BN; p.TN = N / BN;
    p.log_bm = BM == 256 ? 8 : 7; p.log_bn = BN == 256 ? 8 : 7;
    p.rLDN = rLDN;
    p.RA = c.RA; p.RE = c.RE; p.cseg = c.cseg_dev; p.G = G; p.gtable = c.group_table; p.MM = c.MM; p.monitor = c.monitor;
    p.stream_deliver = c.deliver && (long long)M * N * 2 >= kStreamDeliverFrom;
    p.D2 = c.deliver; p.deliver_from = c.deliver_from; p.gstart = c.group_start;
    p.nslices = c.nslices; p.slice_first = c.slice_first; p.slice_count = c.slice_count;

    if (mode != kPlain) {
        if (!c.MM || !c.RA || !c.cseg_dev) return fail(FO_ERR_ARG, "fo_gemm_signal: null MM/RA/cSeg");
        if (G <= 0) return fail(FO_ERR_ARG, "fo_gemm_signal: G=%d", G);
        const int T = (M / BM) * (N / BN);
        if (rLDN <= 0 || T % rLDN) return fail(FO_ERR_SHAPE, "fo_gemm_signal: rLDN=%d must divide the %d tiles", rLDN, T);
        if (mode == kScatter && !c.RE) return fail(FO_ERR_ARG, "fo_gemm_scatter: null RE");
        if (c.deliver && (c.deliver_from < 0 || c.deliver_from > T))
            return fail(FO_ERR_ARG, "fo_gemm_launch: deliver_from=%d outside 0..%d", c.deliver_from, T);
        if (c.deliver && c.monitor) return fail(FO_ERR_ARG, "fo_gemm_launch: monitor tickets are taken by signalled tiles; nothing may be delivered");
        if (c.deliver && mode == kScatter) {
            if (!c.group_table || !c.group_start) return fail(FO_ERR_ARG, "fo_gemm_launch: a delivered scatter needs group_table and group_start");
            if (rLDN != 1) return fail(FO_ERR_SHAPE, "fo_gemm_launch: a delivered scatter needs rLDN 1, got %d", rLDN);
            if (c.nslices <= 0 || BM % c.nslices) return fail(FO_ERR_SHAPE, "fo_gemm_launch: %d slices of a tile of %d rows", c.nslices, BM);
            if (c.slice_first < 0 || c.slice_count <= 0 || c.slice_first + c.slice_count > c.nslices)
                return fail(FO_ERR_ARG, "fo_gemm_launch: slices [%d, %d) outside 0..%d", c.slice_first, c.slice_first + c.slice_count, c.nslices);
            if (c.slice_count > 1 && (c.slice_stride < 0 || c.slice_stride % BN))
                return fail(FO_ERR_SHAPE, "fo_gemm_launch: slice_stride=%lld is not a whole number of rows of %d", c.slice_stride, BN);
            p.slice_rows = (int)(c.slice_stride / BN);
        }
    }
    // in place: one store of each element is enough
    if (mode == kSignal && c.deliver == D && c.deliver_from == 0) keep_d = false;
    if (!keep_d) p.D = nullptr;
    if ((uintptr_t)c.deliver & 15) return fail(FO_ERR_ARG, "fo_gemm: operands must be 16-byte aligned");
    if (is_skinny(c)) return launch_skinny(dtype, M, N, K, A, B, D, c.deliver, N, false, timer, stream);
    const DeviceFacts* facts;
    if (int e = device_facts(&facts)) return e;
    Plan plan;
    if (int e = plan_for(c, ask || c.workspace, facts->cus, &plan)) return e;
    void* workspace = c.workspace;
    bool enough = c.workspace_bytes >= plan.bytes;
    if (ask && plan.bytes) {
        workspace = nullptr;
        if (int e = ask(context, plan.bytes, &workspace)) return e;
        enough = workspace != nullptr;
    }
    if (plan.bytes && !enough)
        if (int e = plan_for(c, false, facts->cus, &plan)) return e;
    p.M = M - plan.strip_m; p.N = N - plan.strip_n;
    // Shapes that are multiples of 128 keep the kernel without row and column predicates (an odd
    // multiple of 128 is half a macro tile, which that kernel handles by whole quadrants).
    const bool edge = any_shape && (p.M % 128 || p.N % 128 || N % 8);
    p.GM = (p.M + plan.macro.m - 1) / plan.macro.m; p.GN = (p.N + plan.macro.n - 1) / plan.macro.n;
    p.gn_magic = raster_magic(p.GN);
    p.split_from = plan.from; p.split_tiles = plan.tiles; p.splits = plan.splits; p.split_panels = plan.panels;
    // A call without a workspace adds in the order of k, in whatever tile.
    p.turn = ask || (c.workspace && enough) ? turn_panels(plan.macro, p.M, p.N, K, facts->cus) : 0;
    if (plan.tiles) {
        if ((uintptr_t)workspace & 15) return fail(FO_ERR_ARG, "fo_gemm: the workspace must be 16-byte aligned");
        p.arrived = (int*)workspace;
        p.partial = (float*)((char*)workspace + FO_WORKSPACE_ZEROED);
    }
    const int macro = plan.macro.m;
    // The event pair of a call of more than one launch spans them all.
    if (plan.strip_m || plan.strip_n) {
        LaunchTimer first;
        std::swap(first.start, timer.start);
        const size_t from = plan.strip_m ? (size_t)p.M * N * 2 : (size_t)p.N * 2;   // of D, in bytes
        void* D2 = c.deliver ? (char*)c.deliver + from : nullptr;
        const int rc = plan.strip_m ? launch_skinny(dtype, plan.strip_m, N, K, (const char*)A + (size_t)p.M * K * 2, B, (char*)D + from, D2, N, false, first, stream)
                                    : launch_skinny(dtype, plan.strip_n, M, K, (const char*)B + (size_t)p.N * K * 2, A, (char*)D + from, D2, N, true, first, stream);
        if (rc != FO_OK) return rc;
    }
    hipEvent_t reduced = nullptr;
    if (plan.tiles && macro != 64) std::swap(reduced, timer.stop);
    // A workgroup that has its CU to itself takes the ring of four panels ahead: nothing else hides the latency of
    // its copies (256x4096x7168, 256 parts: 25.3 us, 22.5; with two on a CU the LDS allows two panels ahead).
    const bool deep = macro == 64 || (macro == 128 && plan.macro.n == 128 && default_forms() && p.split_from + p.split_tiles * p.splits <= facts->cus);
    int rc;
    if (plan.macro.n != macro) rc = launch_gemm_tall(mode, dtype, edge, p, timer, stream);
    else if (deep) rc = launch_gemm_deep(macro, mode, dtype, edge, p, timer, stream);
    else if (dtype == FO_F16)
        rc = macro == 256 ? launch_mt<_Float16, 256>(mode, edge, p, timer, stream) : launch_mt<_Float16, 128>(mode, edge, p, timer, stream);
    else
        rc = macro == 256 ? launch_mt<__bf16, 256>(mode, edge, p, timer, stream) : launch_mt<__bf16, 128>(mode, edge, p, timer, stream);
    if (rc == FO_OK && plan.tiles && macro != 64) rc = launch_split_reduce(mode, dtype, macro, p, reduced, stream);
    return rc;
}

int gemm_rounds(int algo, int M, int N, int* per_round, int* last_first) {
    int BM, BN, BK;
    if (!per_round || !last_first) return fail(FO_ERR_ARG, "fo_gemm_rounds: null output");
    if (algo_tile(algo, &BM, &BN, &BK) != FO_OK) return fail(FO_ERR_ARG, "fo_gemm_rounds: Algo %d out of range", algo);
    if (M <= 0 || N <= 0 || M % BM || N % BN) return fail(FO_ERR_SHAPE, "fo_gemm_rounds: M=%d N=%d vs tile %dx%d", M, N, BM, BN);
    const DeviceFacts* facts;
    if (int e = device_facts(&facts)) return e;
    const Macro t = hint_macro(BM, BN, M, N);
    const long long total = (long long)((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n);
    const long long at_once = (long long)facts->cus * (t.m == 256 ? 1 : 2);   // workgroups a CU holds: LDS
    const long long T = (long long)(M / BM) * (N / BN);   // half macro tiles at the edges make the slots approximate: hints
    *per_round = (int)((T * at_once + total - 1) / total);
    *last_first = (int)((T * ((total - 1) / at_once * at_once) + total - 1) / total);
    return FO_OK;
}

int raster_hint(int algo, int M, int N, int* hint) {
    int BM, BN, BK;
    if (algo_tile(algo, &BM, &BN, &BK) != FO_OK) return fail(FO_ERR_ARG, "fo_raster_hint: Algo %d out of range", algo);
    if (!hint) return fail(FO_ERR_ARG, "fo_raster_hint: null hint");
    if (M <= 0 || N <= 0 || M % BM || N % BN) return fail(FO_ERR_SHAPE, "fo_raster_hint: M=%d N=%d vs tile %dx%d", M, N, BM, BN);
    const Macro t = hint_macro(BM, BN, M, N);
    const int GM = (M + t.m - 1) / t.m, GN = (N + t.n - 1) / t.n, TM = M / BM, TN = N / BN;
    const int tiles_m = t.m / BM, tiles_n = t.n / BN;
    int k = 0;
    for (int pid = 0; pid < GM * GN; ++pid) {
        const TileCoord c = t.m > t.n ? raster_order<kGroupM / 2, kUnitN * 2>(pid, GM, GN, raster_magic(GN))
                                      : raster_order(pid, GM, GN, raster_magic(GN));
        for (int i = 0; i < tiles_m; ++i)
            for (int j = 0; j < tiles_n; ++j) {
                const int tm = c.m * tiles_m + i, tn = c.n * tiles_n + j;
                if (tm < TM && tn < TN) hint[k++] = tm * TN + tn;   // half macro tiles at the matrix edge
            }
    }
    return FO_OK;
}

int tune(const char* key, int value) {
    if (!key) return fail(FO_ERR_ARG, "fo_tune: null key");
    if (!set_knob(key, value)) return fail(FO_ERR_ARG, "fo_tune: unknown knob '%s' or value %d out of its range", key, value);
    return FO_OK;
}

}  // namespace fo
