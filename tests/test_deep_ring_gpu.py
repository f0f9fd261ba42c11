"""The GEMM with four panels ahead (64x64 tiles, and 128x128 ones that have a CU to themselves) and with three (256x128):
K from less than one panel to more than a full turn of the rings (of three and four slots: twelve panels), whole and partial last panels, tiles whole and cut, against exact
sums.  The operands are small whole numbers, so every fp32 sum is exact and the result is its rounding."""
import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi

pytestmark = pytest.mark.gpu


def _object():
    flashoverlap_amd.load()
    o = torch.classes.flashoverlap_class.OverlapImpl()
    o.mccl_init(0, 1, torch.ops.flashoverlap_op.generate_mccl_id())
    o.mutlass_init()
    o.overlap_init()
    return o


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("macro", [0, 128, 256128])   # 0: 64x64 at these sizes
@pytest.mark.parametrize("k", [8, 64, 72, 128, 192, 200, 256, 264, 320, 384, 576, 632, 768, 776, 1088, 1672])
def test_every_length_of_k(k, macro, dtype):
    o = _object()
    g = torch.Generator().manual_seed(k)
    for m, n in [(128, 256), (64, 128), (101, 203), (300, 136)]:
        a = torch.randint(-3, 4, (m, k), generator=g)
        b = torch.randint(-3, 4, (n, k), generator=g)
        want = (a.double() @ b.double().t()).to(dtype)
        A, B = a.to(dtype).cuda(), b.to(dtype).cuda()
        C = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        try:
            assert capi.lib().fo_tune(b"macro_tile", macro) == 0
            for _ in range(3):
                o.mutlass_gemm(A, B, C, 1)
                torch.cuda.synchronize()
                assert torch.equal(C.cpu(), want), (m, n, k)
        finally:
            capi.lib().fo_tune(b"macro_tile", 0)
