"""The workspace of GEMMs that are split over K: an object makes it where it can, and a call for which it cannot
be made is computed without.  Integer-valued inputs: split or not, the result is the same bit for bit."""
import ctypes

import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi

pytestmark = pytest.mark.gpu

M, N, K = 4225, 4104, 1984     # 17 x 17 macro tiles of 256x256, the 33 behind a whole round in parts: the largest workspace


def _step(m, n, k):
    """Which of the workspaces of 4, 16 and 64 MiB a plain call takes."""
    c = capi.GemmCall(mode=0, dtype=capi.FO_BF16, algo=1, M=m, N=n, K=k, rLDN=1, nslices=1)
    need = ctypes.c_size_t()
    capi.check(capi.lib().fo_gemm_workspace(ctypes.byref(c), ctypes.byref(need)))
    return need.value and sum(need.value > 4096 + (s << 20) for s in (4, 16)) + 1


@pytest.fixture
def call(dev):
    """A plain GEMM on an object and a stream of its own, and what it has to give."""
    flashoverlap_amd.load()
    assert _step(M, N, K) == 3
    gen = torch.Generator().manual_seed(19)
    A, B = (torch.randint(-2, 3, (r, K), generator=gen).to(torch.bfloat16).to(dev) for r in (M, N))
    want = (A.float() @ B.float().t()).to(torch.bfloat16).cpu()     # compared there: one of the tests leaves the device no memory
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        o = torch.classes.flashoverlap_class.OverlapImpl()
        o.mutlass_init()
        C = torch.empty(M, N, dtype=torch.bfloat16, device=dev)

    def run():
        C.zero_()
        torch.cuda.synchronize()
        run.launch()
        torch.cuda.synchronize()
        return run.right()

    run.stream, run.launch, run.right = stream, lambda: o.mutlass_gemm(A, B, C, 1), lambda: torch.equal(C.cpu(), want)
    return run


def test_no_memory_for_the_workspace(call):
    def reserved():
        return torch.cuda.memory_reserved() / torch.cuda.get_device_properties(0).total_memory

    ooms = torch.cuda.memory_stats()["num_ooms"]
    with torch.cuda.stream(call.stream):
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction(reserved())
        try:
            assert call() and call()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.cuda.memory_stats()["num_ooms"] == ooms + 1    # asked for once
        assert call()


def test_first_call_from_another_stream(call):
    """torch's current stream is not the GEMM's when the workspace is made."""
    before = torch.cuda.memory_stats(0)["allocation.all.allocated"]
    assert torch.cuda.current_stream() != call.stream
    call.launch()
    assert torch.cuda.memory_stats(0)["allocation.all.allocated"] > before
    torch.cuda.synchronize()
    assert call.right() and call()


def test_first_call_while_another_stream_is_captured(call):
    """The GEMM's stream is not the one that is captured: the call runs at once, and takes no memory."""
    graph = torch.cuda.CUDAGraph()
    other = torch.cuda.Stream()
    x = torch.zeros(1024, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=other, capture_error_mode="thread_local"):
        x.add_(1)
        made = torch.cuda.memory_stats()["allocation.all.allocated"]
        call.launch()
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == made
    torch.cuda.synchronize()
    assert call.right()
    for _ in range(2):
        graph.replay()
        assert call()
    assert (x == 2).all()


def test_threads_on_one_object(dev):
    """Plain calls of several threads on one object, the first ones at the same time, with workspaces of two sizes."""
    import threading
    flashoverlap_amd.load()
    gen = torch.Generator().manual_seed(23)
    shapes = [(256, 4096, 7168), (128, 1024, 4096)]
    assert [_step(*s) for s in shapes] == [2, 1]
    work = []
    for m, n, k in shapes:
        A, B = (torch.randint(-2, 3, (r, k), generator=gen).to(torch.bfloat16).to(dev) for r in (m, n))
        work.append((A, B, (A.float() @ B.float().t()).to(torch.bfloat16)))
    outs = [[torch.zeros(m, n, dtype=torch.bfloat16, device=dev) for m, n, _ in shapes] for _ in range(8)]
    o = torch.classes.flashoverlap_class.OverlapImpl()
    o.mutlass_init()
    torch.cuda.synchronize()
    start, failed = threading.Barrier(len(outs)), []

    def worker(mine, first):
        try:
            start.wait()
            for i in range(20):
                s = (first + i) % 2
                o.mutlass_gemm(work[s][0], work[s][1], mine[s], 1)
        except Exception as e:
            failed.append(e)

    threads = [threading.Thread(target=worker, args=(mine, t % 2)) for t, mine in enumerate(outs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    assert all(torch.equal(c, w[2]) for mine in outs for c, w in zip(mine, work))
