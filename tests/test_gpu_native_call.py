"""The native call path (csrc/sq_torch.cpp): it follows a matrix whose tensors change, leaves to Python what it does not cover,
holds what it hands to the library, runs on the current stream, and its op raises in backward."""

import copy
import sys
import threading

import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import _Workspace, linear_small
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


def test_second_thread_replaces_workspace_and_matrices():
    """Calls of one thread while another replaces the shared workspace by larger ones and sets attributes of the matrices: what a
    call was handed stays its own until it has launched (results stay right, tensors allocated meanwhile are not written to)."""
    ps = core.PackedShards([to_device(synth(96, 1024, 8, 16, seed=1)), to_device(synth(300, 1024, 8, 16, seed=2))])
    x = rand_x(2, 1024, torch.bfloat16, seed=3).cuda()
    want, dev = ps.forward(x), x.device
    size, others = _Workspace.get(1, dev).numel(), []
    called, replaced, ys = threading.Semaphore(0), [], []

    def replace():
        for k in range(1, 25):
            if not called.acquire(timeout=60):                  # (one replacement per call at least, beside the calls that follow)
                return
            _Workspace.get(size + (k << 20), dev)               # (same stream: torch's default one on both threads)
            ps.rls[k & 1].row_scale = ps.rls[k & 1].row_scale.clone()
            others.append(torch.full((size + (k << 20),), 7, dtype=torch.uint8, device=dev))
            replaced.append(len(ys))

    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-5)
    try:
        t = threading.Thread(target=replace)
        t.start()
        while t.is_alive() and len(ys) < 20000:
            ys.append(ps.forward(x))
            called.release()
        t.join()
    finally:
        sys.setswitchinterval(interval)
    assert len(replaced) == 24 and replaced[0] >= 1 and len(ys) >= 24
    assert all(torch.equal(y, want) for y in ys[:: max(1, len(ys) // 200)] + ys[-1:])
    assert all(bool((o == 7).all()) for o in others)


def test_calls_on_a_second_stream():
    ps = core.PackedShards([to_device(synth(96, 512, 8, 16, seed=1)), to_device(synth(40, 512, 8, 16, seed=2))])
    x = rand_x(3, 512, torch.bfloat16, seed=3).cuda()
    want, side = ps.forward(x), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        ys = [_lib.native().forward(ps, x) for _ in range(3)]
    torch.cuda.synchronize()
    assert all(torch.is_tensor(y) and torch.equal(y, want) for y in ys)


def test_outgrown_workspace_waits_for_the_stream_that_used_it():
    dev, side = torch.device("cuda", torch.cuda.current_device()), torch.cuda.Stream()
    size = 24 << 20
    old = _Workspace.get(size, dev, "other streams").data_ptr()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)                          # stands for a product on the old buffer
        _Workspace.get(2 * size, dev, "other streams")
    assert torch.empty(size, dtype=torch.uint8, device=dev).data_ptr() != old
    torch.cuda.synchronize()
    del _Workspace.bufs[(str(dev), "other streams")]
