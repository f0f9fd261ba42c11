"""fo_build_group_tables: the slot -> group table and the groups' first slots, against the linear scan, with
empty groups, more groups than the workgroup has threads, and slots beyond the last group."""
import numpy as np
import pytest
import torch

from flashoverlap_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,high", [(1, 1), (1, 2048), (2, 1024), (13, 98), (63, 3), (64, 5), (65, 5), (1023, 2), (1024, 4),
                                    (1025, 4), (5000, 3)])
@pytest.mark.parametrize("beyond", [0, 1, 1500])
def test_tables(G, high, beyond):
    rng = np.random.default_rng(G + beyond)
    cseg = rng.integers(0, high + 1, G).astype(np.int32)
    cseg[rng.integers(G)] = high
    ends = np.cumsum(cseg)
    T = int(ends[-1]) + beyond
    want = np.minimum(np.searchsorted(ends, np.arange(T), side="right"), G - 1)
    L, dev = capi.lib(), torch.device("cuda")
    cs = torch.from_numpy(cseg).to(dev)
    table = torch.full((T + 8,), -7, dtype=torch.int32, device=dev)
    start = torch.full((G + 8,), -7, dtype=torch.int32, device=dev)
    capi.check(L.fo_build_group_tables(cs.data_ptr(), G, T, table.data_ptr(), start.data_ptr(), None))
    torch.cuda.synchronize()
    assert np.array_equal(table.cpu().numpy(), np.concatenate([want, np.full(8, -7)]))
    assert np.array_equal(start.cpu().numpy(), np.concatenate([ends - cseg, np.full(8, -7)]))
    table.fill_(-7)
    capi.check(L.fo_build_group_table(cs.data_ptr(), G, T, table.data_ptr(), None))
    torch.cuda.synchronize()
    assert np.array_equal(table.cpu().numpy()[:T], want)
