// Host orchestration of the overlapped path on one MI355X.  Follows the call
// structure of the reference's src/overlap_impl.cu (GEMM on the caller's
// stream, a per-group wait -> collective loop on a second stream, an event
// join back), with the collective replaced by a consumer copy into a staging
// buffer and every failure reported through TORCH_CHECK instead of exit().
#include "overlap_impl.h"

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>

#include <exception>
#include <map>

#include "host_common.h"

// Copies made while the GEMM runs use non-temporal stores once a call makes this many bytes
// of them: c3 (33 MB) is 1.5 % faster with ordinary stores, c5 (100 MB) 2.5 % and c4 (201 MB)
// 4-8 % faster with non-temporal ones.
static constexpr size_t kStreamCopiesFrom = 64u << 20;

// Longest K with which the GEMM's epilogue delivers all groups: a choice, see groups_to_wait_for.
static constexpr int kDeliverAllK = 8192;

OverlapImpl::OverlapImpl() = default;

OverlapImpl::~OverlapImpl() {
    if (comm_stream_) fo_stream_destroy(comm_stream_);
}

void OverlapImpl::MutlassInit() {
    // Like the reference, the stream that is current now is used for every
    // later GEMM of this object (src/overlap_impl.cu:38-40).
    gemm_stream_ = (void*)c10::hip::getCurrentHIPStream().stream();
    gemm_ready_ = true;
}

void OverlapImpl::McclInit(int64_t tp_rank, int64_t tp_size, std::vector<int64_t> tp_id) {
    TORCH_CHECK(tp_size >= 1 && tp_rank >= 0 && tp_rank < tp_size, "mccl_init: rank ", tp_rank, " of ", tp_size);
    TORCH_CHECK(tp_id.size() == 16, "mccl_init: the id must have 16 entries, got ", tp_id.size());
    // One GPU: no communicator is created (the reference also skips it for
    // size 1, src/overlap_impl.cu:65-68).  A size above 1 only selects the
    // ReduceScatter slicing that a rank of that world would see.
    my_rank_ = tp_rank;
    my_size_ = tp_size;
}

void OverlapImpl::OverlapInit() {
    if (!comm_stream_) FO_CALL(fo_stream_create(&comm_stream_));
}

void OverlapImpl::SetConsumerMode(int64_t mode) {
    TORCH_CHECK(mode >= 0 && mode <= 2, "set_consumer_mode: 0 (auto), 1 (per group) or 2 (persistent), got ", mode);
    consumer_mode_ = mode;
}

void OverlapImpl::SetConsumerBlocks(int64_t blocks) {
    int cus = 0;
    FO_CALL(fo_device_info(&cus, nullptr, nullptr));
    // The persistent consumer's workgroups wait beside the GEMM's: at most one per CU.
    TORCH_CHECK(blocks >= 1 && blocks <= cus, "set_consumer_blocks: 1..", cus, " (one workgroup per CU), got ", blocks);
    consumer_blocks_ = blocks;
}

int OverlapImpl::consumer_blocks() {
    if (consumer_blocks_ == 0) {   // default: one workgroup per CU
        int cus = 0;
        FO_CALL(fo_device_info(&cus, nullptr, nullptr));
        consumer_blocks_ = cus;
    }
    return (int)consumer_blocks_;
}

void OverlapImpl::SetWaitTimeoutMs(int64_t ms) {
    TORCH_CHECK(ms >= 1 && ms <= 3600 * 1000, "set_wait_timeout_ms: 1..3600000, got ", ms);
    FO_CALL(fo_set_wait_timeout_ms((int)ms));
}

// The word this object's waits count their expiries in (one int32 on the device of `like`).
int* OverlapImpl::expired_word(const at::Tensor& like) {
    if (!expired_.defined() || expired_.device() != like.device()) {
        expired_ = at::zeros({1}, like.options().dtype(at::kInt));
        // once per object: the fill runs on torch's current stream, the waits on another one
        c10::hip::getCurrentHIPStream().synchronize();
    }
    return expired_.data_ptr<int>();
}

int64_t OverlapImpl::WaitTimeouts(bool reset) {
    if (!expired_.defined()) return 0;   // no overlapped call has run yet
    c10::DeviceGuard guard(expired_.device());
    if (comm_stream_) FO_CALL(fo_stream_sync(comm_stream_));
    if (gemm_ready_) FO_CALL(fo_stream_sync(gemm_stream_));
    const int64_t n = expired_.item<int>();
    if (reset && n) expired_.zero_();
    return n;
}

void OverlapImpl::SetCheckTimeouts(bool on) { check_timeouts_ = on; }

// Checked mode: wait for the call to finish and turn an expired wait into an
// error.  The counters then hold partial counts, which would make every later
// wait on them expire too (or pass at once), so they are cleared here.
void OverlapImpl::raise_on_timeout(at::Tensor& MM, const char* who) {
    if (!check_timeouts_) return;
    FO_CALL(fo_stream_sync(gemm_stream_));   // the call's join has ordered it behind the second stream
    const int n = expired_.item<int>();
    if (n == 0) return;
    expired_.zero_();
    MM.zero_();
    TORCH_CHECK(false, who, ": ", n, " bounded wait(s) expired before their group completed; the consumer's output "
                "is incomplete and MM has been zeroed (a cSeg that does not match the tiles, or a GEMM slower than the "
                "wait timeout)");
}

at::Tensor OverlapImpl::Staging() const {
    TORCH_CHECK(staging_.defined(), "staging: no all-reduce style call has run yet");
    return staging_;
}

void OverlapImpl::SetStaging(at::Tensor buffer) {
    TORCH_CHECK(buffer.defined() && buffer.is_cuda() && buffer.is_contiguous(),
                "set_staging: the buffer must be a contiguous GPU tensor");
    TORCH_CHECK(buffer.scalar_type() == at::kHalf || buffer.scalar_type() == at::kBFloat16,
                "set_staging: the buffer must be float16 or bfloat16, got ", buffer.scalar_type());
    staging_ = buffer.view({buffer.numel()});
}

void OverlapImpl::require_gemm() const {
    TORCH_CHECK(gemm_ready_, "OverlapImpl: call mutlass_init() first");
}

void OverlapImpl::require_overlap() const {
    require_gemm();
    TORCH_CHECK(comm_stream_ != nullptr, "OverlapImpl: call overlap_init() first");
}

at::Tensor& OverlapImpl::staging_like(const at::Tensor& C) {
    if (!staging_.defined() || staging_.numel() != C.numel() || staging_.scalar_type() != C.scalar_type() ||
        staging_.device() != C.device())
        staging_ = at::empty({C.numel()}, C.options());
    return staging_;
}

const int* OverlapImpl::group_table_for(const at::Tensor& cseg_cpu, const at::Tensor& cseg_gpu, int T) {
    const int G = (int)cseg_cpu.numel();
    const int* host = cseg_cpu.data_ptr<int>();
    std::vector<int> key(host, host + G);
    key.push_back(T);
    const bool same_device = group_table_.defined() && group_table_.device() == cseg_gpu.device();
    if (!same_device || key != table_key_) {
        group_table_ = at::empty({T}, cseg_gpu.options());
        group_start_ = at::empty({G}, cseg_gpu.options());
        FO_CALL(fo_build_group_tables(cseg_gpu.data_ptr<int>(), G, T, group_table_.data_ptr<int>(),
                                      group_start_.data_ptr<int>(), gemm_stream_));
        table_key_ = std::move(key);
    }
    return group_table_.data_ptr<int>();
}

void OverlapImpl::bulk_consume(const void* src, void* dst, size_t bytes) {
    FO_CALL(fo_consume(src, dst, bytes, gemm_stream_));
}

static fo_gemm_call describe(int mode, const fo_host::GemmShape& s, int64_t algo, int64_t rLDN, const at::Tensor& A,
                             const at::Tensor& B, const at::Tensor& C, const at::Tensor& RA, bool monitor) {
    fo_gemm_call c{};
    c.mode = mode;
    c.dtype = s.dtype;
    c.algo = (int)algo;
    c.M = s.M;
    c.N = s.N;
    c.K = s.K;
    c.rLDN = (int)rLDN;
    c.A = A.data_ptr();
    c.B = B.data_ptr();
    c.D = C.defined() ? C.data_ptr() : nullptr;
    c.RA = RA.defined() ? RA.data_ptr<int>() : nullptr;
    c.monitor = monitor ? 1 : 0;
    c.nslices = 1;
    return c;
}

std::shared_ptr<SplitWorkspace> SplitWorkspace::of_stream(int device, void* stream) {
    static std::mutex mutex;
    static std::map<std::pair<int, void*>, std::weak_ptr<SplitWorkspace>> pool;
    std::lock_guard<std::mutex> lock(mutex);
    for (auto it = pool.begin(); it != pool.end();) it = it->second.expired() ? pool.erase(it) : std::next(it);
    std::weak_ptr<SplitWorkspace>& slot = pool[{device, stream}];
    std::shared_ptr<SplitWorkspace> w = slot.lock();
    if (!w) slot = w = std::make_shared<SplitWorkspace>();
    return w;
}

// The GEMM, with a workspace if its shape can use one.
// A captured call runs unsplit: its graph may be replayed beside later calls on this stream, after this
// object is gone and any number of times, so neither the stream's workspace nor memory that is given back
// when the call returns may be written by it, and nothing here lives as long as the graph.
void OverlapImpl::launch_gemm(const fo_gemm_call& call, const at::Tensor& like) {
    struct Request {   // the workspace that the library asked for is this call's until its kernels are enqueued
        OverlapImpl* self;
        const at::Tensor* like;
        std::shared_ptr<SplitWorkspace> w;
        std::unique_lock<std::mutex> lock;
        std::exception_ptr error;
    } request{this, &like, nullptr, {}, nullptr};
    const auto provide = [](void* context, size_t bytes, void** out) noexcept -> int {
        Request& r = *(Request*)context;
        try {
            *out = r.self->workspace_of(bytes, *r.like, r.w, r.lock);
            return FO_OK;
        } catch (...) {
            r.error = std::current_exception();
            return FO_ERR_HIP;
        }
    };
    const int rc = fo_gemm_run(&call, call.D != nullptr, provide, &request, gemm_stream_);   // (no D: a layer that returns what is delivered)
    if (request.error) std::rethrow_exception(request.error);
    FO_CALL(rc);
}

void* OverlapImpl::workspace_of(size_t need, const at::Tensor& like, std::shared_ptr<SplitWorkspace>& w,
                                std::unique_lock<std::mutex>& lock) {
    int step = 0;
    while (step < 3 && need > FO_WORKSPACE_ZEROED + ((size_t)4 << 20 << 2 * step)) ++step;
    if (step == 3) return nullptr;
    int capturing = 0;
    FO_CALL(fo_stream_is_capturing(gemm_stream_, &capturing));
    if (capturing) return nullptr;
    w = workspace_on(like.device().index());
    lock = std::unique_lock<std::mutex>(w->mutex);
    if (!w->buffer[step].defined()) make_workspace(*w, like, step, FO_WORKSPACE_ZEROED + ((int64_t)4 << 20 << 2 * step));
    return w->buffer[step].defined() ? w->buffer[step].data_ptr() : nullptr;
}

// This object's hold on the workspace of its GEMM stream.  Threads may launch on one object at the same time.
std::shared_ptr<SplitWorkspace> OverlapImpl::workspace_on(int device) {
    std::lock_guard<std::mutex> lock(workspace_mutex_);
    if (!workspace_ || workspace_device_ != device || workspace_stream_ != gemm_stream_) {
        workspace_ = SplitWorkspace::of_stream(device, gemm_stream_);
        workspace_device_ = device;
        workspace_stream_ = gemm_stream_;
    }
    return workspace_;
}

// The workspace only makes a call faster.  Where the device has no memory for it the call runs without, and
// so do the later ones of that size on this stream: an allocation that fails first gives all cached memory back
// and waits for the device, which must not happen on every call, and a shape keeps its order of additions.
void OverlapImpl::make_workspace(SplitWorkspace& w, const at::Tensor& like, int step, int64_t bytes) {
    if (w.refused[step]) return;
    // Taking memory can mean a hipMalloc, which would end a capture of the current stream (the GEMM's own is not
    // being captured, launch_gemm): the next call makes the buffer.
    int capturing = 0;
    FO_CALL(fo_stream_is_capturing((void*)c10::hip::getCurrentHIPStream().stream(), &capturing));
    if (capturing) return;
    // made and cleared on the GEMM's stream, whichever is current
    c10::hip::HIPStreamGuard on(c10::hip::getStreamFromExternal((hipStream_t)gemm_stream_, like.device().index()));
    at::Tensor made;
    try {
        made = at::empty({bytes}, like.options().dtype(at::kByte));
    } catch (const c10::OutOfMemoryError&) {
        w.refused[step] = true;
        return;
    }
    made.narrow(0, 0, FO_WORKSPACE_ZEROED).zero_();
    w.buffer[step] = std::move(made);
}

static bool shares_memory(const void* p, int64_t elems, const void* dst, int64_t dst_elems) {
    return (const char*)dst < (const char*)p + 2 * elems && (const char*)p < (const char*)dst + 2 * dst_elems;
}
static bool inside_output(const fo_gemm_call& c, const void* dst, int64_t dst_elems) {
    return shares_memory(c.D, (int64_t)c.M * c.N, dst, dst_elems);
}

// Whether the GEMM's epilogue may write the receive buffer: not if it shares memory with an operand, which
// other workgroups still read, nor with C, whose rows other workgroups write (a rank's receive buffer can
// be the first rows of C: a copy that starts when its group is complete writes rows of groups that are
// complete too).  C itself as the buffer of an all-reduce is no such case: both stores of an element are
// made by one lane, to one address, with one value.
static bool can_deliver(const fo_gemm_call& c, const void* dst, int64_t dst_elems) {
    if (shares_memory(c.A, (int64_t)c.M * c.K, dst, dst_elems) || shares_memory(c.B, (int64_t)c.N * c.K, dst, dst_elems))
        return false;
    return !inside_output(c, dst, dst_elems) || (dst == c.D && c.mode != FO_GEMM_SCATTER);
}

void OverlapImpl::Gemm(at::Tensor A, at::Tensor B, at::Tensor C, int64_t Algo) {
    require_gemm();
    const fo_host::GemmShape s = fo_host::check_gemm(A, B, C, "mutlass_gemm");
    c10::DeviceGuard guard(A.device());
    fo_gemm_call call = describe(FO_GEMM_PLAIN, s, Algo, 1, A, B, C, at::Tensor(), false);
    launch_gemm(call, C);
}

// Called before the GEMM is enqueued.  While the caller's stream is being captured into a
// graph, the communication stream's part of the call is first ordered behind the caller's
// stream (not behind the GEMM, which comes later): the capture then follows the work onto the
// second stream, and with the join at the end the call is a closed fork/join pattern of
// kernels.  Outside a capture the fork is left out, as in the reference: the event it puts in
// front of the GEMM costs 5-9 us of every call.
// Ahead of the GEMM launch of an overlapped call: the word its waits count their expiries in
// exists (creating it waits for the stream once per object, which must not happen between the
// GEMM and its waiters), and checked mode is not combined with a capture.
void OverlapImpl::prepare_call(const at::Tensor& MM, const char* who) {
    refuse_checked_capture(who);
    expired_word(MM);
}

// Checked mode ends every call with a wait for the stream, which a capture forbids (it would
// invalidate the capture and leave the caller with an unrelated error).
void OverlapImpl::refuse_checked_capture(const char* who) {
    if (!check_timeouts_) return;
    int capturing = 0;
    FO_CALL(fo_stream_is_capturing(gemm_stream_, &capturing));
    TORCH_CHECK(!capturing, who, ": set_check_timeouts(true) makes the call wait for its own completion, which is not "
                "allowed while the stream is being captured into a graph; turn it off for captured calls and read "
                "wait_timeouts() after a replay instead");
}

void OverlapImpl::fork_comm_stream(int waited, int G) {
    if (waited == 0 || (waited == G && G <= 1 && consumer_mode_ != 2)) return;   // the second stream is not used
    int capturing = 0;
    FO_CALL(fo_stream_is_capturing(gemm_stream_, &capturing));
    if (capturing) FO_CALL(fo_stream_join(gemm_stream_, comm_stream_));
}

// How many of the groups are released through their counters; the others are delivered by the
// GEMM's epilogue.  A group's wait and copy overlap with the GEMM only if the group completes
// before the GEMM does.  The last group never does, and neither do the groups whose tiles all
// belong to the last round of workgroups: their copies used to start when the GEMM had ended, one
// wait and one copy launch after the other (sixteen groups of one round, 4096x4096x4096: 140 us
// behind a GEMM of 97).  The epilogue has these tiles in registers and stores them twice instead.
//
// With K of up to kDeliverAllK it does so for every group.  The copy of an early group reads again what the
// epilogue had in registers, and its traffic costs the GEMM beside it more than the second store does.  Call with
// norm, early groups copied / all delivered, bf16 unless said, us: 7424x6016x640 141 / 110, 3840x7808x880 105 / 78,
// 8192x4096x512 93 / 66, 12288x8192x1024 290 / 255, 16384x8192x1024 385 / 359, reducescatter 15104x1280x2936 fp16 in a
// world of two 160 / 140.  The longer a round the better the copies hide: 8192x8192x8192 791 / 787, 8192x8192x16384
// 1549 / 1542, level.  So the limit is no crossing, at which one of the two becomes the slower: it is a choice, within
// the lengths at which neither costs anything.  Above it groups are released as they complete, which is what lets a
// consumer start early; below, a caller who wants that takes an explicit mode.
// Checked mode and monitor mode keep every group on its counter (the first reports a count that
// does not come out, the second takes its tickets from the signals), and so do the explicit modes.
int OverlapImpl::groups_to_wait_for(const fo_gemm_call& call, const int* cseg, int nslices, int* first_slot,
                                    int* per_round) {
    int BM, BN, BK, late = 0;
    FO_CALL(fo_algo_tile(call.algo, &BM, &BN, &BK));
    if (consumer_mode_ != 0 || check_timeouts_ || call.monitor || BM % nslices) return call.G;
    if (call.K <= kDeliverAllK) return 0;
    FO_CALL(fo_gemm_rounds(call.algo, call.M, call.N, per_round, &late));
    int g = 0, slot = 0;
    while (g + 1 < call.G && slot < late) slot += cseg[g++];
    *first_slot = slot;
    return g;
}

// Release of the first `waited` groups (the others have been delivered by the GEMM itself): the
// reference's host loop (one wait kernel and one consumer launch per group,
// src/overlap_impl.cu:257-265 / 312-323), the same with one pair of launches for the groups of a round
// (per_round slots), or one persistent kernel that does the walk on the device.  On return the GEMM
// stream is ordered behind every group's copy.
//
// Groups of one round fill their counters at the same moment, and a pair of launches of their own
// each then only queues up, on the host too: 15104x1280x2936 fp16 in 13 groups of 98 tiles took 222 us
// with its norm, 133 of them of the host, and takes 165; 7424x6016x640 in 5 of 302 148 -> 130, 9856x6400x1408
// in 14 of 275 253 -> 230.  It also leaves the automatic mode without the persistent kernel, of which
// two (of two objects, on two streams) can hold the registers that a GEMM they wait for needs.
//
// in_order: dst lies in C, and a group's copy writes where an earlier group's is read from: the copies
// follow each other, the last one too.
void OverlapImpl::consume_groups(const at::Tensor& C, void* dst, int64_t tile_elems, const at::Tensor& cseg_cpu,
                                 const at::Tensor& cseg_gpu, at::Tensor& MM, int waited, int per_round,
                                 int nslices, int64_t slice_stride, bool in_order) {
    const int G = (int)cseg_cpu.numel();
    const int* cseg = cseg_cpu.data_ptr<int>();
    const int slice_first = slice_stride ? 0 : (int)my_rank_;      // stride 0: only this rank's slice
    const int slice_count = slice_stride ? nslices : 1;
    int* expired = expired_.data_ptr<int>();   // this object's own count of expired waits (prepare_call)
    if (consumer_mode_ == 2) {
        FO_CALL(fo_wait_consume(cseg_gpu.data_ptr<int>(), waited, MM.data_ptr<int>(), C.data_ptr(), dst, tile_elems,
                                nslices, slice_first, slice_count, slice_stride, nullptr, consumer_blocks(),
                                expired, comm_stream_));
        // The caller's stream continues only after the last group is consumed
        // (src/overlap_impl.cu:267-270).
        FO_CALL(fo_stream_join(comm_stream_, gemm_stream_));
        return;
    }
    const size_t esz = C.element_size();
    const char* src = (const char*)C.data_ptr();
    // The groups before the last are copied while the GEMM runs: if that is a lot of data,
    // with stores that leave the GEMM's operands in the memory-side cache.
    int64_t beside = 0;
    for (int g = 0; g < waited && g + 1 < G; ++g) beside += tile_elems * cseg[g] / nslices * slice_count * (int64_t)esz;
    const int beside_policy = beside >= (int64_t)kStreamCopiesFrom ? FO_COPY_STREAM : FO_COPY_CACHED;
    int64_t acc = 0;
    for (int g = 0; g < waited; ++g) {
        // If the last group of the call is among them (explicit modes, checked and monitor mode): it
        // completes with the GEMM, so nothing is left for it to overlap with, and
        // it is released on the GEMM's own stream, where stream order stands in for the wait
        // kernel (the counter is settled by the copy launch itself), and the groups before it,
        // finished long ago on the communication stream, are joined behind it.  A last group
        // on the communication stream would instead put a fresh cross-stream dependency
        // (10-20 us on this platform) between its copy and the caller's next kernel.
        const bool last = g == G - 1;
        void* stream = last ? gemm_stream_ : comm_stream_;
        if (last && in_order && g > 0) FO_CALL(fo_stream_join(comm_stream_, gemm_stream_));
        const int64_t comm = tile_elems * cseg[g];
        // the groups up to `end` complete in the round in which this one does
        int end = g + 1;
        int64_t tiles = cseg[g];
        if (per_round)
            while (end < waited && end + 1 < G && (int64_t)(end - g + 1) * slice_count < 65536 &&
                   (acc / tile_elems + tiles + cseg[end] - 1) / per_round == (acc / tile_elems + cseg[g] - 1) / per_round)
                tiles += cseg[end++];
        if (end > g + 1) {
            FO_CALL(fo_wait_groups(cseg_gpu.data_ptr<int>(), g, end - g, MM.data_ptr<int>(), expired, stream));
            FO_CALL(fo_consume_groups(cseg_gpu.data_ptr<int>(), group_start_.data_ptr<int>(), g, end - g, src, dst, tile_elems,
                                      nslices, slice_first, slice_count, slice_stride, beside_policy,
                                      tile_elems * tiles * esz / nslices * slice_count, stream));
            acc += tile_elems * tiles;
            g = end - 1;
            continue;
        }
        if (!last) FO_CALL(fo_wait(cseg[g], MM.data_ptr<int>() + g, expired, stream));
        // One launch per group, like the one collective call per group of the reference: this
        // rank's slice of the group, or all ranks' slices into their receive buffers side by side.
        const int64_t part = comm / nslices;
        FO_CALL(fo_consume_slices(cseg[g], last ? MM.data_ptr<int>() + g : nullptr,
                                  src + (acc + slice_first * part) * esz, (char*)dst + (acc / nslices) * esz,
                                  part * esz, slice_count, slice_stride * esz,
                                  last ? FO_COPY_CACHED : beside_policy, expired, stream));
        acc += comm;
    }
    // The caller's stream continues only after every group is consumed (src/overlap_impl.cu:267-270).
    if (waited > 1 || waited < G) FO_CALL(fo_stream_join(comm_stream_, gemm_stream_));
}

// What the overlapped calls share: the GEMM (call.mode, RE and nslices say which) and the
// release of its groups into dst.  C undefined: it is not kept, and is made only if groups are copied out of it.
void OverlapImpl::overlapped_call(fo_gemm_call& call, const fo_host::SignalShape& g, at::Tensor C, const at::Tensor& out,
                                  const at::Tensor& cseg_cpu, const at::Tensor& cseg_gpu, at::Tensor& MM,
                                  int64_t slice_stride, const char* who) {
    prepare_call(MM, who);
    void* dst = out.data_ptr();
    call.cseg_dev = cseg_gpu.data_ptr<int>();
    call.G = g.G;
    call.MM = MM.data_ptr<int>();
    const int64_t kept = (int64_t)call.M * call.N / (slice_stride ? 1 : call.nslices);
    int per_round = 0;
    const int waited = can_deliver(call, dst, kept) ? groups_to_wait_for(call, cseg_cpu.data_ptr<int>(), call.nslices,
                                                                         &call.deliver_from, &per_round)
                                                    : g.G;
    released_ = waited;
    if (waited || call.mode == FO_GEMM_SCATTER) {   // (an all-reduce that signals nothing looks no group up)
        call.group_table = group_table_for(cseg_cpu, cseg_gpu, g.T);
        call.group_start = group_start_.data_ptr<int>();
    }
    if (waited < g.G) {
        call.deliver = dst;
        call.slice_first = slice_stride ? 0 : (int)my_rank_;
        call.slice_count = slice_stride ? call.nslices : 1;
        call.slice_stride = slice_stride;
    }
    if (!C.defined() && waited) {
        C = at::empty({call.M, call.N}, out.options());
        call.D = C.data_ptr();
    }
    fork_comm_stream(waited, g.G);
    launch_gemm(call, out);
    if (waited == 0) return;
    consume_groups(C, dst, (int64_t)g.BM * g.BN, cseg_cpu, cseg_gpu, MM, waited, per_round, call.nslices, slice_stride,
                   inside_output(call, dst, kept));
    raise_on_timeout(MM, who);
}

// An all-reduce into `out` (defined here unless C's staging buffer is to be it), a ReduceScatter into D.
void OverlapImpl::allreduce_call(const at::Tensor& A, const at::Tensor& B, const at::Tensor& C, const at::Tensor& out,
                                 at::Tensor& MM, const at::Tensor& RA, int64_t rLDN, const at::Tensor& cSEG_CPU,
                                 const at::Tensor& cSEG_GPU, int64_t Algo, bool if_monitor) {
    require_overlap();
    const char* who = "gemm_allreduce_overlap";
    const fo_host::GemmShape s = fo_host::check_gemm(A, B, C, who, !out.defined());
    const fo_host::SignalShape g =
        fo_host::check_signal(s, MM, RA, at::Tensor(), rLDN, cSEG_CPU, cSEG_GPU, (int)Algo, if_monitor, 1, who);
    c10::DeviceGuard guard(A.device());
    fo_gemm_call call = describe(FO_GEMM_SIGNAL, s, Algo, rLDN, A, B, C, RA, if_monitor);
    overlapped_call(call, g, C, out.defined() ? out : staging_like(C), cSEG_CPU, cSEG_GPU, MM, 0, who);
}

void OverlapImpl::reducescatter_call(const at::Tensor& A, const at::Tensor& B, const at::Tensor& C, bool keeps_c,
                                     const at::Tensor& D, at::Tensor& MM, const at::Tensor& RA, const at::Tensor& RE,
                                     int64_t rLDN, const at::Tensor& cSEG_CPU, const at::Tensor& cSEG_GPU, int64_t Algo,
                                     bool if_monitor) {
    require_overlap();
    const char* who = "gemm_reducescatter_overlap";
    const fo_host::GemmShape s = fo_host::check_gemm(A, B, C, who, keeps_c);
    const fo_host::SignalShape g =
        fo_host::check_signal(s, MM, RA, RE, rLDN, cSEG_CPU, cSEG_GPU, (int)Algo, if_monitor, (int)my_size_, who);
    const int64_t total = (int64_t)s.M * s.N;
    fo_host::check_buffer(D, A, who, "D");
    // D is one rank's receive buffer [M/ws, N] as in the reference, or all ws
    // of them stacked [ws, M/ws, N].
    TORCH_CHECK(D.numel() == total / my_size_ || D.numel() == total, who,
                ": D must hold M*N/world_size = ", total / my_size_, " or M*N = ", total, " elements, got ", D.numel());
    c10::DeviceGuard guard(A.device());
    fo_gemm_call call = describe(FO_GEMM_SCATTER, s, Algo, rLDN, A, B, C, RA, if_monitor);
    call.RE = RE.data_ptr<int>();
    call.nslices = (int)my_size_;
    const int64_t stride = (D.numel() == total && my_size_ > 1) ? total / my_size_ : 0;
    overlapped_call(call, g, C, D, cSEG_CPU, cSEG_GPU, MM, stride, who);
}

void OverlapImpl::GemmAllReduceOverlap(at::Tensor A, at::Tensor B, at::Tensor C, at::Tensor MM, at::Tensor RA,
                                       int64_t rLDN, at::Tensor cSEG_CPU, at::Tensor cSEG_GPU, int64_t Algo,
                                       bool if_monitor) {
    allreduce_call(A, B, C, at::Tensor(), MM, RA, rLDN, cSEG_CPU, cSEG_GPU, Algo, if_monitor);
}

void OverlapImpl::GemmReduceScatterOverlap(at::Tensor A, at::Tensor B, at::Tensor C, at::Tensor D, at::Tensor MM,
                                           at::Tensor RA, at::Tensor RE, int64_t rLDN, at::Tensor cSEG_CPU,
                                           at::Tensor cSEG_GPU, int64_t Algo, bool if_monitor) {
    reducescatter_call(A, B, C, true, D, MM, RA, RE, rLDN, cSEG_CPU, cSEG_GPU, Algo, if_monitor);
}

// The layers' calls return what is delivered and keep no C: where every group is delivered none is made or stored (call
// with norm, C stored / not, us: all-reduce 8192x8192x1024 182 / 168, 3840x7552x2688 154 / 148; reducescatter 3072x6528x536 of
// eight ranks 41.7 / 39.3, 8192x4096x2048 of two 122 / 118; the smallest calls by the allocation, 15.6 / 15.2).
at::Tensor OverlapImpl::AllReduceLinear(at::Tensor A, at::Tensor B, at::Tensor MM, at::Tensor RA, at::Tensor cSEG_CPU,
                                        at::Tensor cSEG_GPU, int64_t Algo) {
    TORCH_CHECK(A.dim() == 2 && B.dim() == 2, "allreduce_linear: A [M,K] and B [N,K] must be 2-D");
    at::Tensor out = at::empty({A.size(0), B.size(0)}, A.options());
    SetStaging(out);
    allreduce_call(A, B, at::Tensor(), out, MM, RA, 1, cSEG_CPU, cSEG_GPU, Algo, false);
    return out;
}

at::Tensor OverlapImpl::ReduceScatterLinear(at::Tensor A, at::Tensor B, at::Tensor MM, at::Tensor RA, at::Tensor RE,
                                            at::Tensor cSEG_CPU, at::Tensor cSEG_GPU, int64_t Algo) {
    TORCH_CHECK(A.dim() == 2 && B.dim() == 2, "reducescatter_linear: A [M,K] and B [N,K] must be 2-D");
    at::Tensor out = at::empty({A.size(0) / my_size_, B.size(0)}, A.options());
    reducescatter_call(A, B, at::Tensor(), false, out, MM, RA, RE, 1, cSEG_CPU, cSEG_GPU, Algo, false);
    return out;
}

// The bulk copy that stands in for the collective starts when the GEMM has ended, so the GEMM's
// epilogue makes it: C is stored twice instead of being read back.
void OverlapImpl::GemmAllReduce(at::Tensor A, at::Tensor B, at::Tensor C, int64_t Algo) {
    require_gemm();
    const fo_host::GemmShape s = fo_host::check_gemm(A, B, C, "gemm_allreduce");
    c10::DeviceGuard guard(A.device());
    fo_gemm_call call = describe(FO_GEMM_PLAIN, s, Algo, 1, A, B, C, at::Tensor(), false);
    void* dst = staging_like(C).data_ptr();
    const bool after = !can_deliver(call, dst, C.numel());
    if (!after) call.deliver = dst;
    launch_gemm(call, C);
    if (after) bulk_consume(C.data_ptr(), dst, C.numel() * C.element_size());
}

void OverlapImpl::GemmReduceScatter(at::Tensor A, at::Tensor B, at::Tensor C, at::Tensor D, int64_t Algo) {
    Gemm(A, B, C, Algo);
    fo_host::check_buffer(D, C, "gemm_reducescatter", "D");
    const int64_t recv = C.numel() / my_size_;
    TORCH_CHECK(D.numel() >= recv, "gemm_reducescatter: D holds ", D.numel(), " elements, needs ", recv);
    c10::DeviceGuard guard(C.device());
    // What this rank would receive (src/overlap_impl.cu:104-107), without the sum over ranks.
    bulk_consume((const char*)C.data_ptr() + my_rank_ * recv * C.element_size(), D.data_ptr(),
                 recv * C.element_size());
}

void OverlapImpl::GemmAll2All(at::Tensor A, at::Tensor B, at::Tensor C, at::Tensor D, int64_t Algo,
                              at::Tensor mLen_CPU) {
    TORCH_CHECK(my_size_ == 1, "gemm_all2all: exchanging rows with ", my_size_ - 1,
                " peers needs more than one GPU, which this build does not drive");
    Gemm(A, B, C, Algo);  // a world of one sends and receives nothing (src/overlap_impl.cu:132-143)
}

void OverlapImpl::McclAllReduce(at::Tensor C) {
    require_gemm();
    fo_host::check_buffer(C, C, "mccl_allreduce", "C");
    c10::DeviceGuard guard(C.device());
    at::Tensor& staging = staging_like(C);
    bulk_consume(C.data_ptr(), staging.data_ptr(), C.numel() * C.element_size());
}

void OverlapImpl::SegAllReduce(at::Tensor C, at::Tensor cSEG_CPU, int64_t SegNum) {
    require_gemm();
    fo_host::check_buffer(C, C, "seg_allreduce", "C");
    TORCH_CHECK(cSEG_CPU.device().is_cpu() && cSEG_CPU.scalar_type() == at::kInt && cSEG_CPU.is_contiguous(),
                "seg_allreduce: cSEG_CPU must be a contiguous int32 host tensor");
    TORCH_CHECK(SegNum > 0 && C.numel() % SegNum == 0, "seg_allreduce: SegNum=", SegNum, " must divide M*N");
    c10::DeviceGuard guard(C.device());
    at::Tensor& staging = staging_like(C);
    const int* cseg = cSEG_CPU.data_ptr<int>();
    const int64_t unit = C.numel() / SegNum;
    int64_t acc = 0;
    // src/overlap_impl.cu:160-173: cSEG_CPU[s] counts units of M*N/SegNum.
    for (int64_t sidx = 0; sidx < cSEG_CPU.numel() && acc < C.numel(); ++sidx) {
        const int64_t n = unit * cseg[sidx];
        TORCH_CHECK(n >= 0 && acc + n <= C.numel(), "seg_allreduce: segments exceed M*N");
        bulk_consume((const char*)C.data_ptr() + acc * C.element_size(),
                     (char*)staging.data_ptr() + acc * C.element_size(), n * C.element_size());
        acc += n;
    }
}

void OverlapImpl::McclReduceScatter(at::Tensor C) {
    require_gemm();
    fo_host::check_buffer(C, C, "mccl_reducescatter", "C");
    c10::DeviceGuard guard(C.device());
    // In place in the reference: the rank's part of C receives the sum
    // (src/overlap_impl.cu:183-186).  Stand-in: that part goes to staging.
    at::Tensor& staging = staging_like(C);
    const int64_t recv = C.numel() / my_size_;
    const size_t off = my_rank_ * recv * C.element_size();
    bulk_consume((const char*)C.data_ptr() + off, (char*)staging.data_ptr() + off, recv * C.element_size());
}

void OverlapImpl::McclAll2All(at::Tensor C, at::Tensor D, at::Tensor mLen_CPU) {
    TORCH_CHECK(my_size_ == 1, "mccl_all2all: exchanging rows with ", my_size_ - 1,
                " peers needs more than one GPU, which this build does not drive");
}
