"""A plain GEMM whose last few rows or columns are computed by the skinny kernel and the rest by macro tiles of whole
multiples of 128."""
import ctypes as C

import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi

pytestmark = pytest.mark.gpu


def _workspace(M, N, K, dtype):
    c = capi.GemmCall(mode=0, dtype=capi.dtype_code(dtype), algo=1, M=M, N=N, K=K, rLDN=1, nslices=1)
    need = C.c_size_t()
    capi.check(capi.lib().fo_gemm_workspace(C.byref(c), C.byref(need)))
    return need.value


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,strip_m,strip_n", [
    (2080, 4096, 4096, 32, 0), (2049, 4096, 4096, 1, 0), (2065, 4091, 4096, 17, 0),   # the last: rows of D unaligned
    (2048, 4097, 4096, 0, 1), (2048, 4128, 4096, 0, 32), (2041, 4104, 4096, 0, 8), (2000, 4115, 4128, 0, 19),
])
def test_rows_and_columns_behind_the_last_whole_tile(M, N, K, strip_m, strip_n, dtype):
    """Small whole numbers: every order of the fp32 additions gives the exact sums.  All of D and of its bulk copy is
    written and nothing around it; called with a workspace and without one."""
    # the plan is that of the shape without the strip
    assert _workspace(M, N, K, dtype) == _workspace(M - strip_m, N - strip_n, K, dtype)
    flashoverlap_amd.load()
    o = torch.classes.flashoverlap_class.OverlapImpl()
    o.mccl_init(0, 1, torch.ops.flashoverlap_op.generate_mccl_id())
    o.mutlass_init()
    o.overlap_init()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = (torch.randint(-2, 3, (r, K), generator=g, device="cuda").to(dtype) for r in (M, N))
    want = (A.float() @ B.float().t()).to(dtype)
    guard = 4096
    bufs = [torch.full((guard + M * N + guard,), 7.0, dtype=dtype, device="cuda") for _ in range(2)]
    c, staging = (b[guard:guard + M * N].view(M, N) for b in bufs)
    o.set_staging(staging)
    for run in (lambda: o.gemm_allreduce(A, B, c, 1),
                lambda: capi.check(capi.lib().fo_gemm(capi.dtype_code(dtype), 1, M, N, K, A.data_ptr(), B.data_ptr(), c.data_ptr(), None))):
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        run()
        torch.cuda.synchronize()
        assert torch.equal(c, want) and torch.equal(staging, want)
        assert all((b[:guard] == 7.0).all() and (b[guard + M * N:] == 7.0).all() for b in bufs)


@pytest.mark.parametrize("M,N,K", [(2080, 4096, 4096), (2048, 4128, 4096), (1024, 2056, 7680)])
def test_timed_call_with_a_strip(dev, M, N, K):
    """The event pair of fo_time_next_launch spans the skinny launch, the tiles' and, of the last shape with its workspace, the
    reduction's; the call is the untimed one."""
    L, dt = capi.lib(), torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(M)
    A, B = (torch.randn(r, K, generator=g, device="cuda").to(dt) for r in (M, N))
    evs = [C.c_void_p() for _ in range(4)]
    for e in evs:
        capi.check(L.fo_event_create(C.byref(e)))
    inner0, inner1, outer0, outer1 = evs
    need = _workspace(M, N, K, dt)
    assert need == _workspace(M - M % 128, N - N % 128, K, dt)     # the strip is taken
    work = torch.zeros(need // 4 + 1, device="cuda")
    got = []
    for timed in (False, True):
        D = torch.zeros(M, N, dtype=dt, device="cuda")
        c = capi.GemmCall(mode=0, dtype=capi.FO_BF16, algo=1, M=M, N=N, K=K, rLDN=1, nslices=1, A=A.data_ptr(), B=B.data_ptr(),
                          D=D.data_ptr(), workspace=work.data_ptr(), workspace_bytes=need)
        torch.cuda.synchronize()
        capi.check(L.fo_event_record(outer0, None))
        if timed:
            capi.check(L.fo_time_next_launch(inner0, inner1))
        capi.check(L.fo_gemm_launch(C.byref(c), None))
        capi.check(L.fo_event_record(outer1, None))
        torch.cuda.synchronize()
        got.append(D)
    assert torch.equal(*got)
    inner, outer = C.c_float(), C.c_float()
    capi.check(L.fo_event_elapsed_ms(inner0, inner1, C.byref(inner)))
    capi.check(L.fo_event_elapsed_ms(outer0, outer1, C.byref(outer)))
    for e in evs:
        capi.check(L.fo_event_destroy(e))
    # the operations of the tiles and the operand that the strip reads, at rates above the chip's peaks
    rest = (M - M % 128) * (N - N % 128)
    least = 2 * rest * K / 2.6e15 + 2 * (N if M % 128 else M) * K / 30e12
    assert least < inner.value * 1e-3 <= outer.value * 1e-3
