"""The overlapped call captured into a graph and replayed.

The reference's call (src/overlap_impl.cu:221-271) starts work on its second
stream without ordering it behind the caller's stream, so stream capture cannot
follow it there.  Here the call forks the second stream off the caller's before
the GEMM and joins it back at the end, which makes GEMM || wait+copy -> RMSNorm
one capturable unit of kernels (no memset nodes, no allocation after the first
call).  Every replay is checked bit for bit against the same call made eagerly,
with new operand values and eager work between the replays."""
import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi, tiling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,mode", [(16, 1), (4, 2)])   # 4 groups released one by one; 16 groups, persistent consumer
def test_overlapped_call_replays_from_a_graph(dev, w, mode):
    flashoverlap_amd.load()
    # a wait that cannot be satisfied (graph branches run in the wrong order) must fail the test, not stall it
    capi.check(capi.lib().fo_set_wait_timeout_ms(2000))
    M, N, K, algo = 1024, 1024, 512, 1
    dt = torch.bfloat16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    T = TM * TN
    cseg = tiling.uniform_cseg(T, w)
    cSeg_CPU = torch.tensor(cseg, dtype=torch.int32)
    cSeg_GPU = cSeg_CPU.to(dev)
    RA = tiling.reorder_indices(T, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    gen = torch.Generator().manual_seed(11)

    def operands():
        return ((torch.randn(M, K, generator=gen) / K ** 0.5).to(dt).to(dev),
                (torch.randn(N, K, generator=gen) / K ** 0.5).to(dt).to(dev))

    side = torch.cuda.Stream()
    try:
        with torch.cuda.stream(side):
            o = torch.classes.flashoverlap_class.OverlapImpl()
            o.mccl_init(0, 1, torch.ops.flashoverlap_op.generate_mccl_id())
            o.mutlass_init()      # the GEMM stream is `side` from here on
            o.overlap_init()
            o.set_consumer_mode(mode)
            A, B = operands()
            W = (1 + 0.1 * torch.randn(N, generator=gen)).to(dt).to(dev)
            C = torch.empty(M, N, dtype=dt, device=dev)
            y = torch.empty(M, N, dtype=dt, device=dev)
            counter = torch.zeros(max(len(cseg), TN), dtype=torch.int32, device=dev)

            def call():
                o.gemm_allreduce_overlap(A, B, C, counter, RA, 1, cSeg_CPU, cSeg_GPU, algo, False)
                torch.ops.flashoverlap_op.reorder_rmsnorm(o.staging().view(M, N), y, W, BM, BN, 1, RA)

            for _ in range(3):    # first calls allocate the staging buffer and the group table
                call()
            side.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                call()
            # checked mode waits for the call's completion, which a capture forbids: refused up front,
            # before anything is enqueued, with an error that says so (capture_error_mode: the failed
            # capture must not poison the streams of the rest of the process)
            o.set_check_timeouts(True)
            refused = torch.cuda.CUDAGraph()
            with pytest.raises(RuntimeError, match="set_check_timeouts"):
                with torch.cuda.graph(refused, stream=side, capture_error_mode="thread_local"):
                    call()
            o.set_check_timeouts(False)
            del refused
            for replay in range(4):
                print(f"graph replay {replay} w={w} mode={mode}", flush=True)
                a_new, b_new = operands()
                A.copy_(a_new)
                B.copy_(b_new)
                call()                                  # eager, same buffers
                side.synchronize()
                want_staging, want_y = o.staging().clone(), y.clone()
                assert want_y.float().abs().sum() > 0
                o.staging().zero_()
                y.zero_()
                C.zero_()
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                assert o.wait_timeouts(True) == 0
                assert counter.cpu().sum() == 0
                assert torch.equal(o.staging(), want_staging)
                assert torch.equal(y, want_y)
    finally:
        capi.check(capi.lib().fo_set_wait_timeout_ms(5000))


@pytest.fixture
def short_waits():
    """A wait that cannot be satisfied (graph branches run in the wrong order) must fail the test, not stall it."""
    capi.check(capi.lib().fo_set_wait_timeout_ms(2000))
    yield
    capi.check(capi.lib().fo_set_wait_timeout_ms(5000))


def _whole_numbers(dev, dt, gen, *shape):
    """Small integers: every sum is exact in fp32, so a call that is split over K and one that is not agree bit for bit."""
    return torch.randint(-2, 3, shape, generator=gen, dtype=torch.int8).to(dev).to(dt)


@pytest.mark.parametrize("M,N,K,w,ws", [
    (1024, 1024, 512, 4, 1),       # every group is delivered by the epilogue
    (128, 4096, 4096, 32, 1),      # split over K when it is not captured, every group delivered
    (128, 4096, 4096, 8, 4),
    (8192, 4352, 64, 100, 1),      # delivered, in three rounds
    (8192, 4352, 8200, 100, 1),    # groups of a round released together on the second stream, the last ones delivered
    (8192, 4352, 8200, 100, 4),
    (4352, 4096, 1544, 200, 1),    # delivered, and sixteen tiles split over K when it is not captured
    (4352, 4096, 8200, 200, 1),    # released, and split
])
def test_default_mode_replays_from_a_graph(dev, short_waits, M, N, K, w, ws):
    """The automatic mode: a warmed call that is captured allocates nothing, and every replay gives what the
    eager call gives, also with eager calls of the same object in between."""
    flashoverlap_amd.load()
    algo, dt = 1, torch.bfloat16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    cseg = tiling.uniform_cseg(TM * TN, w)
    cs = torch.tensor(cseg, dtype=torch.int32)
    cs_gpu = cs.to(dev)
    RA = tiling.reorder_indices(TM * TN, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev) if ws > 1 else None
    gen = torch.Generator().manual_seed(13)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        o = torch.classes.flashoverlap_class.OverlapImpl()
        o.mccl_init(ws - 1, ws, torch.ops.flashoverlap_op.generate_mccl_id())
        o.mutlass_init()
        o.overlap_init()
        A, B = _whole_numbers(dev, dt, gen, M, K), _whole_numbers(dev, dt, gen, N, K)
        W = (1 + 0.1 * torch.randn(N, generator=gen)).to(dt).to(dev)
        C, recv, y = (torch.zeros(rows, N, dtype=dt, device=dev) for rows in (M, M // ws, M // ws))
        counter = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
        o.set_staging(recv)

        def call():
            if ws > 1:
                o.gemm_reducescatter_overlap(A, B, C, recv, counter, RA, RE, 1, cs, cs_gpu, algo, False)
            else:
                o.gemm_allreduce_overlap(A, B, C, counter, RA, 1, cs, cs_gpu, algo, False)
            torch.ops.flashoverlap_op.reorder_rmsnorm(recv, y, W, BM // ws, BN, 1, RA)

        for _ in range(2):
            call()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            made = torch.cuda.memory_stats()["allocation.all.allocated"]
            call()
            assert torch.cuda.memory_stats()["allocation.all.allocated"] == made
        assert (o.released_groups() > 0) == (K > 8192)     # the captured call's
        for replay in range(3):
            print(f"graph replay {replay} {M}x{N}x{K} w={w} ws={ws}", flush=True)
            A.copy_(_whole_numbers(dev, dt, gen, M, K))
            call()
            side.synchronize()
            want = [t.clone() for t in (C, recv, y)]
            assert want[2].float().abs().sum() > 0
            for t in (C, recv, y):
                t.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert o.wait_timeouts(True) == 0 and not counter.any()
            assert all(torch.equal(t, w_) for t, w_ in zip((C, recv, y), want))


def test_capture_that_torch_does_not_see(dev):
    """A capture begun through the runtime on torch's current stream: torch's allocator knows nothing of it and
    hands memory that is given back inside it to the next tensor.  The graph may write to nothing but C."""
    import ctypes
    flashoverlap_amd.load()
    L, dt = capi.lib(), torch.bfloat16
    M, N, K = 128, 4096, 4096       # split over K when it is not captured
    gen = torch.Generator().manual_seed(17)
    side = torch.cuda.Stream()
    stream = ctypes.c_void_p(side.cuda_stream)
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    with torch.cuda.stream(side):
        o = torch.classes.flashoverlap_class.OverlapImpl()
        o.mutlass_init()
        A, B = _whole_numbers(dev, dt, gen, M, K), _whole_numbers(dev, dt, gen, N, K)
        C = torch.zeros(M, N, dtype=dt, device=dev)
        o.mutlass_gemm(A, B, C, 1)
        side.synchronize()
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        assert L.hipStreamBeginCapture(stream, 2) == 0       # relaxed
        o.mutlass_gemm(A, B, C, 1)
        assert L.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
        assert L.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
        others = [torch.full((n << 18,), 7.0, device=dev) for n in (4, 16, 17, 64) for _ in range(2)]
        for replay in range(3):
            print(f"raw graph replay {replay}", flush=True)
            A.copy_(_whole_numbers(dev, dt, gen, M, K))
            want = (A.float() @ B.float().t()).to(dt)
            C.zero_()
            assert L.hipGraphLaunch(run, stream) == 0
            side.synchronize()
            assert torch.equal(C, want)
            assert all((t == 7.0).all() for t in others)
            o.mutlass_gemm(A, B, C, 1)                       # eager, split
            assert torch.equal(C, want)
        side.synchronize()
        assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
