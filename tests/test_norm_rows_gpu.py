"""RMSNorm at the row lengths where the kernel changes (a wavefront, four or eight wavefronts and 1 to 16
chunks per thread, two passes), one element group on either side, few and many rows, plain and reorder with
the shift-only gather and the general one.  Oracle and bar of the other norm tests: two storage ulps."""
import numpy as np
import pytest
import torch

from flashoverlap_amd import capi
from oracle import fo_oracle as O

pytestmark = pytest.mark.gpu


def _close(got, ref, dt):
    ulp = 2 ** -10 if dt == torch.float16 else 2 ** -7
    assert ((got.float() - ref.float()).abs() <= 2 * ulp * ref.float().abs() + 1e-6).all()


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bs,dim", [(5, 2048), (3, 2056), (130, 4096), (7, 4104), (3, 6144), (9, 6152), (2, 8200),
                                    (3, 12296), (2, 16384), (1, 16392), (2, 32768), (1, 32776), (1, 65536), (1, 65544)])
def test_plain(fo_lib, dev, dt, bs, dim):
    g = torch.Generator().manual_seed(dim + bs)
    x, gamma = torch.randn(bs, dim, generator=g).to(dt), (1 + 0.1 * torch.randn(dim, generator=g)).to(dt)
    buf = torch.full((64 + bs * dim + 64,), 7.0, dtype=dt, device=dev)
    dx, dg = x.to(dev), gamma.to(dev)
    capi.check(fo_lib.fo_rmsnorm(capi.dtype_code(dt), dx.data_ptr(), dg.data_ptr(), buf[64:].data_ptr(), bs, dim, 1e-5, None))
    torch.cuda.synchronize()
    _close(buf[64:64 + bs * dim].cpu().view(bs, dim), O.rmsnorm(x, gamma, 1e-5), dt)
    assert (buf[:64] == 7.0).all() and (buf[64 + bs * dim:] == 7.0).all()


@pytest.mark.parametrize("bs,dim,BM,BN,rldn", [(64, 2048, 16, 128, 1), (32, 2176, 16, 128, 1), (64, 4096, 64, 8, 1),
                                               (24, 4224, 8, 128, 1), (36, 6144, 12, 256, 1), (16, 8192, 16, 128, 2),
                                               (16, 16640, 16, 128, 1), (8, 65536, 8, 256, 1)])
def test_reorder(fo_lib, dev, bs, dim, BM, BN, rldn):
    dt = torch.bfloat16
    g = torch.Generator().manual_seed(dim + bs)
    cn, gamma = torch.randn(bs, dim, generator=g).to(dt), (1 + 0.1 * torch.randn(dim, generator=g)).to(dt)
    T = (bs // BM) * (dim // BN)
    ra = O.reorder_indices(T, np.random.default_rng(T).permutation(T))
    x = O.place_tiles(cn, ra, BM, BN, rldn)
    out = torch.empty(bs, dim, dtype=dt, device=dev)
    dx, dg, dra = x.to(dev), gamma.to(dev), torch.from_numpy(ra).to(dev)
    capi.check(fo_lib.fo_reorder_rmsnorm(capi.dtype_code(dt), dx.data_ptr(), dg.data_ptr(), out.data_ptr(), bs, dim, BM,
                                         BN, rldn, dra.data_ptr(), 1e-6, None))
    torch.cuda.synchronize()
    _close(out.cpu(), O.rmsnorm(cn, gamma, 1e-6), dt)
