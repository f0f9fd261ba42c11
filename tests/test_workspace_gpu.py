"""The workspace of GEMMs that are split over K: an object makes it where it can, and a call for which it cannot
be made is computed without.  Integer-valued inputs: split or not, the result is the same bit for bit."""
import pytest
import torch

import flashoverlap_amd

pytestmark = pytest.mark.gpu

M, N, K = 128, 4096, 7168      # 32 tiles in 8 parts of 64 KiB: the workspace is the largest one, 64 MiB


@pytest.fixture
def call(dev):
    """A plain GEMM on an object and a stream of its own, and what it has to give."""
    flashoverlap_amd.load()
    gen = torch.Generator().manual_seed(19)
    A, B = (torch.randint(-2, 3, (r, K), generator=gen).to(torch.bfloat16).to(dev) for r in (M, N))
    want = (A.float() @ B.float().t()).to(torch.bfloat16)
    torch.cuda.synchronize()
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

    run.stream, run.launch, run.right = stream, lambda: o.mutlass_gemm(A, B, C, 1), lambda: torch.equal(C, want)
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
    shapes = [(128, 4096, 7168), (128, 1024, 4096)]
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
