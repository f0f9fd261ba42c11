"""The plain GEMM for up to 32 rows of A: every count of row blocks, N at and around the 16 rows of a
workgroup and on both sides of the change of its size, K of less than a turn, of a ragged last turn and
of more turns than the wavefronts share.  Integer-valued inputs, exact, guard words around both outputs."""
import ctypes as C

import pytest
import torch

from flashoverlap_amd import capi

pytestmark = pytest.mark.gpu
GUARD = 64


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(1, 8), (16, 64), (17, 1096), (130, 4104), (4096, 512), (4101, 72), (4112, 1032)])
def test_skinny_gemm(dev, dt, M, N, K):
    print(f"skinny {dt} {M}x{N}x{K}", flush=True)
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    A, B = (torch.randint(-2, 3, (r, K), generator=g).to(dt).to(dev) for r in (M, N))
    want = (A.float() @ B.float().t()).to(dt)
    buf = torch.full((2, GUARD + M * N + GUARD + -M * N % 8), 7.0, dtype=dt, device=dev)   # both rows 16-byte aligned
    D, D2 = (b[GUARD:GUARD + M * N] for b in buf)
    c = capi.GemmCall(mode=0, dtype=capi.dtype_code(dt), algo=1, M=M, N=N, K=K, rLDN=1, A=A.data_ptr(), B=B.data_ptr(),
                      D=D.data_ptr(), nslices=1, deliver=D2.data_ptr())
    capi.check(capi.lib().fo_gemm_launch(C.byref(c), None))
    torch.cuda.synchronize()
    assert torch.equal(D.view(M, N), want) and torch.equal(D2.view(M, N), want)
    assert (buf[:, :GUARD] == 7.0).all() and (buf[:, GUARD + M * N:] == 7.0).all()
