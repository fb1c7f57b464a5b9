"""Dense decode of matrices with column orders: every output type bit-exact with rows taken one by one and in pairs of one order,
pairs that span orders, a last row alone, row ranges; stacks in one launch with the fp16 copy of x."""

import numpy as np
import pytest
import torch

from oracle import sq_oracle as O
from quantexperiments_amd.kernels import dequant_stack
from tests.helpers import rand_x, synth, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,C,d,bits,G,M", [(1, 8, 8, 16, 1, 2), (3, 4, 4, 8, 1, 3), (70, 2568, 8, 12, 1, 40), (261, 1000, 4, 10, 3, 5), (18, 5120, 8, 16, 2, 4),
                                            (9, 8200, 8, 9, 1, 2), (13, 4100, 4, 12, 1, 6), (5, 16384, 8, 16, 1, 3), (4, 32768, 8, 16, 1, 2),
                                            (2051, 64, 8, 8, 1, 200), (2048, 100, 4, 8, 3, 2)])
def test_dense_decode_is_bit_exact(R, C, d, bits, G, M):
    s = synth(R, C, d, bits, G, M, seed=R + C)
    lin, w = to_device(s, stream=False), s.decode()
    assert np.array_equal(lin.dense(torch.float32).cpu().numpy(), w)
    assert np.array_equal(lin.dense(torch.float16).float().cpu().numpy(), O.round_fp16(w))
    assert np.array_equal(lin.dense(torch.bfloat16).float().cpu().numpy(), O.round_bf16(w))
    for r0, r1 in ((0, R - R // 4), (R // 3, R)):
        assert np.array_equal(lin.dense(torch.float16, rows=(r0, r1)).float().cpu().numpy(), O.round_fp16(w[r0:r1]))


# pairs of rows, pieces of an odd count; one row at a time; more pieces than a launch takes; pieces without orders, in one launch and
# one by one with the copy in a launch of its own; mixed kinds
@pytest.mark.parametrize("R,forms", [(301, [(8, 8, 1, 3)] * 8), (37, [(8, 16, 1, 3)] * 3), (7, [(8, 12, 1, 2)] * 11), (50, [(4, 12, 2, 1)] * 2),
                                     (9, [(8, 16, 1, 1)] * 2), (20, [(8, 16, 1, 3), (4, 10, 1, 3), (8, 16, 1, 1)])])
@pytest.mark.parametrize("T", [0, 1, 77])
def test_stack_and_copy(R, forms, T):
    ss = [synth(R + i % 2, 320, *f, seed=i) for i, f in enumerate(forms)]
    lins = [to_device(s, stream=False) for s in ss]
    out = torch.full((sum(s.R for s in ss), 320), float("nan"), dtype=torch.float16, device="cuda")
    x = rand_x(T, 328, torch.bfloat16, seed=T).cuda()[:, :320] if T else None
    xh = dequant_stack(lins, out, x)
    assert np.array_equal(out.float().cpu().numpy(), np.concatenate([O.round_fp16(s.decode()) for s in ss]))
    assert xh is None if x is None else torch.equal(xh, x.to(torch.float16))
