"""The emulator's torch operators without a GPU: both register with their
schemas, and their fake-tensor rules and the registered autograd formula
give the shapes and dtypes of the network's output and of every parameter
gradient (FakeTensorMode runs no kernel)."""
import ctypes

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


def test_ops_register_and_trace():
    from exoplasim_amd import radiation as r

    f = r.emulator_op()
    fwd = torch.ops.exoplasim_amd.lw_mlp_forward.default._schema
    bwd = torch.ops.exoplasim_amd.lw_mlp_backward.default._schema
    assert len(fwd.arguments) == 9 and len(fwd.returns) == 8
    assert len(bwd.arguments) == 12 and len(bwd.returns) == 8
    with FakeTensorMode():
        x = torch.empty(96, r.NIN)
        ps = []
        for nin, nout in r.LAYERS:
            ps += [torch.empty(nout, nin, requires_grad=True),
                   torch.empty(nout, requires_grad=True)]
        y = f(x, *ps)
        assert y.shape == (96, r.NOUT) and y.dtype == torch.float32
        y.sum().backward()
        for p in ps:
            assert p.grad is not None and p.grad.shape == p.shape


@pytest.mark.parametrize("shape", [(5, 20), (5, 22), (4,), (5, 2), (5, 0)])
def test_backward_refuses_wrong_gradients(monkeypatch, shape):
    """an output gradient that does not broadcast to (rows, 21) raises and
    reaches no kernel, which would read past its end; one that does is read
    broadcast"""
    from exoplasim_amd import radiation as r

    r.emulator_op()
    seen = []

    class Native:
        @staticmethod
        def exo_mlp_train_work(m, backward):
            return 16

        @staticmethod
        def exo_mlp_train_backward(m, gy, *rest):
            seen.append(list((ctypes.c_float * (m * r.NOUT)).from_address(gy)))
            return 0

    monkeypatch.setattr(r, "_proto", lambda: Native)
    monkeypatch.setattr(r, "_stream", lambda: None)
    f32, bf = torch.float32, torch.bfloat16

    def backward(gy):
        m = gy.shape[0]
        return torch.ops.exoplasim_amd.lw_mlp_backward(
            gy, torch.zeros(m, r.KIN, dtype=bf), *[torch.zeros(m, r.NHID) for _ in range(3)],
            *[torch.zeros(m, r.NHID, dtype=bf) for _ in range(3)],
            *[torch.zeros(nout, nin) for nin, nout in r.LAYERS])

    with pytest.raises(RuntimeError):
        backward(torch.ones(shape))
    assert not seen
    col = torch.arange(5, dtype=f32)[:, None]
    for gy in (col, col.double(), col.expand(5, r.NOUT)):
        backward(gy)
        assert seen.pop() == [float(i) for i in range(5) for _ in range(r.NOUT)]
