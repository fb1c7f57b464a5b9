"""Dense decode of d = 4 matrices from a codebook in LDS: every output type bit-exact, with one and several codebooks up to the
largest LDS takes, one chunk pair per row, row ranges, and a stack decoded in one launch with the fp16 copy of x."""

import numpy as np
import pytest
import torch

from oracle import sq_oracle as O
from quantexperiments_amd.kernels import linear_gemm
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,C,bits,G", [(1, 8, 8, 1), (3, 64, 1, 1), (515, 8, 12, 1), (70, 3584, 12, 4), (129, 1000, 10, 2), (40, 896, 14, 1), (9, 264, 5, 16)])
def test_dense_decode_is_bit_exact(R, C, bits, G):
    s = synth(R, C, 4, bits, G, 1, seed=R + C)
    lin, w = to_device(s, stream=False), s.decode()
    assert np.array_equal(lin.dense(torch.float32).cpu().numpy(), w)
    assert np.array_equal(lin.dense(torch.float16).float().cpu().numpy(), O.round_fp16(w))
    assert np.array_equal(lin.dense(torch.bfloat16).float().cpu().numpy(), O.round_bf16(w))
    r0, r1 = R // 3, R - R // 4
    if r1 > r0:
        assert np.array_equal(lin.dense(torch.float32, rows=(r0, r1)).cpu().numpy(), w[r0:r1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("G", [1, 4])
def test_stack_decoded_in_one_launch(dtype, G):
    ss = [synth(R, 192, 4, 12, G, 1, seed=R) for R in (300, 17, 1)]
    x = rand_x(600, 192, dtype, seed=G)
    y = torch.empty(600, 318, dtype=torch.float32, device="cuda")
    linear_gemm([to_device(s) for s in ss], x.cuda(), y)
    ref = np.concatenate([x.float().numpy().astype(np.float64) @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.cpu().numpy(), ref) < 1e-3
