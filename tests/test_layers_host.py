"""The nn.Module wrappers' host logic, with a recorder in the place of the native object."""
from types import SimpleNamespace

import pytest
import torch

from flashoverlap_amd import layers


class _Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append((name, len(args)))


@pytest.mark.parametrize("comm_op,other", [("all_reduce", "reduce_scatter"), ("reduce_scatter", "all_reduce")])
def test_forward_follows_comm_op_and_the_object(monkeypatch, comm_op, other):
    """forward calls the method that `comm_op` names when it runs, on the object that the layer holds then."""
    monkeypatch.setattr(layers.flashoverlap_amd, "load", lambda: None)
    monkeypatch.setattr(layers.torch, "classes",
                        SimpleNamespace(flashoverlap_class=SimpleNamespace(OverlapImpl=_Recorder)))
    cfg = {"BM": 128, "BN": 128, "Algo": 1, "hint": [0, 1, 2, 3], "cSeg": [2, 2]}
    layer = layers.OverlapRowParallelLayer(0, 2, 64, 256, 256, cfg, comm_op, mccl_id=[0] * 16, device="cpu")
    called = {"all_reduce": ("allreduce_linear", 7), "reduce_scatter": ("reducescatter_linear", 8)}
    x = torch.zeros(256, 64, dtype=torch.float16)
    for op in (comm_op, other, comm_op):
        layer.comm_op = op
        layer(x)
        assert layer.overlap_class.calls[-1] == called[op]
    layer.overlap_class = _Recorder()
    layer(x)
    assert layer.overlap_class.calls == [called[comm_op]]
