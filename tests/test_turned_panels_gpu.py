"""Whole tiles of 48 panels and more, whose workgroups begin at eight places of K: one panel less, 48, and counts that eight does and
does not divide, a K with a partial last panel (which begins at the first), in every macro tile, with ragged rows and columns and
signalled.  The operands are small whole numbers, so that every fp32 sum is exact and the result is its rounding."""
import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi, tiling

pytestmark = pytest.mark.gpu


def _object():
    flashoverlap_amd.load()
    o = torch.classes.flashoverlap_class.OverlapImpl()
    o.mccl_init(0, 1, torch.ops.flashoverlap_op.generate_mccl_id())
    o.mutlass_init()
    o.overlap_init()
    return o


def _operands(m, n, k, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a, b = (torch.randint(-3, 4, (r, k), generator=g, device=dev).to(dtype) for r in (m, n))
    return a, b, (a.float() @ b.float().t()).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("macro", [0, 128, 256128, 256])
@pytest.mark.parametrize("k", [3008, 3072, 3080, 3136, 3520, 4096])
def test_every_panel_is_multiplied_once(k, macro, dtype, dev):
    o = _object()
    try:
        assert capi.lib().fo_tune(b"macro_tile", macro) == 0
        for m, n in [(2048, 2048), (1027, 1544), (300, 4095)]:
            a, b, want = _operands(m, n, k, dtype, dev)
            c = torch.full((m, n), float("nan"), dtype=dtype, device=dev)
            o.mutlass_gemm(a, b, c, 1)
            assert torch.equal(c, want), (m, n)
    finally:
        capi.lib().fo_tune(b"macro_tile", 0)


@pytest.mark.parametrize("consumer", [0, 1])   # delivered by the epilogue; released and copied
@pytest.mark.parametrize("m,n,k,algo", [(1280, 2176, 3136, 1), (2560, 2304, 3072, 4), (4352, 4352, 3200, 0)])
def test_signalled_tiles(m, n, k, algo, consumer, dev):
    o, dtype = _object(), torch.bfloat16
    o.set_consumer_mode(consumer)
    a, b, want = _operands(m, n, k, dtype, dev)
    bm, bn, _ = capi.algo_tile(algo)
    tm, tn = m // bm, n // bn
    cseg = tiling.uniform_cseg(tm * tn, 50)
    ra = tiling.reorder_indices(tm * tn, tiling.raster_hint(m, n, algo), dev).reshape(tm, tn)
    cseg_cpu = torch.tensor(cseg, dtype=torch.int32)
    counters = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    c, staging = (torch.full((m, n), float("nan"), dtype=dtype, device=dev) for _ in range(2))
    o.set_staging(staging)
    o.gemm_allreduce_overlap(a, b, c, counters, ra, 1, cseg_cpu, cseg_cpu.to(dev), algo, False)
    torch.cuda.synchronize()
    placed = torch.empty(tm * tn, bm, bn, dtype=dtype, device=dev)
    placed[ra.flatten().long()] = want.reshape(tm, bm, tn, bn).transpose(1, 2).reshape(tm * tn, bm, bn)
    assert torch.equal(c.flatten(), placed.flatten()) and torch.equal(staging.flatten(), placed.flatten())
    assert int(counters.abs().sum()) == 0
