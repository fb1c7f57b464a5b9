"""The native call path (csrc/sq_torch.cpp): it follows a matrix whose tensors change, leaves to Python what it does not cover,
and its op raises in backward."""

import copy

import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import linear_small
from quantexperiments_amd.vllm_ext import core
from tests.helpers import rand_x, synth, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,bits,M", [(8, 16, 1), (8, 16, 3), (4, 12, 1)])
def test_native_call_follows_its_matrices(d, bits, M):
    ps = core.PackedShards([to_device(synth(96, 512, d, bits, 1, M, seed=1)), to_device(synth(40, 512, d, bits, 1, M, seed=2))])
    x = rand_x(3, 512, torch.bfloat16, seed=3).cuda()
    ps.forward(x)                                               # (grows the workspace: a first call may go through Python)
    y = _lib.native().forward(ps, x)
    assert torch.is_tensor(y) and y.shape == (3, 136)
    for z in (x.view(3, 1, 512), x[1]):
        assert torch.equal(_lib.native().forward(ps, z).reshape(-1, 136), ps.forward(z.reshape(-1, 512)))
    a = ps.rls[0]
    twin = copy.deepcopy(a)                                     # (what the native path keeps is not part of the state)
    a.row_scale = a.row_scale * 2
    assert torch.equal(ps.forward(x)[:, :96], y[:, :96] * 2) and torch.equal(ps.forward(x)[:, 96:], y[:, 96:])
    a.row_scale.data = (a.row_scale / 4).data
    assert torch.equal(ps.forward(x)[:, :96], y[:, :96] / 2)
    assert torch.equal(linear_small([twin], x, torch.empty(3, 96, dtype=x.dtype, device="cuda")), y[:, :96])
    # not covered: another dtype, a strided input, no rows, a mismatch (whose error Python words)
    for z in (x.float(), x.repeat(1, 2)[:, ::2], x[:0], x[:, :-8]):
        assert _lib.native().forward(ps, z) == 1
    with pytest.raises(ValueError):
        linear_small(ps.rls, x, torch.empty(3, 100, dtype=x.dtype, device="cuda"))


def test_op_runs_without_gradients_only():
    ps = core.PackedShards([to_device(synth(32, 256, 4, 12, seed=4))])
    h = core.register(ps)
    x = rand_x(2, 256, torch.bfloat16, seed=5).cuda().requires_grad_()
    y = torch.ops.shapequant.linear(x, h)
    assert torch.equal(y.detach(), ps.forward(x.detach()))
    with pytest.raises(NotImplementedError):
        y.sum().backward()
