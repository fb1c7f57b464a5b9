"""The matrix-core decode kernel with its codebooks in LDS, at the splits of a row over waves and workgroups that its plan makes: one
wave and sixteen, short and split rows, idle rounds in the last wave, room for 8 tokens at a time only, two token tiles."""

import numpy as np
import pytest
import torch

from quantexperiments_amd.kernels import linear_small
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,bits,G", [(64, 8, 1), (128, 12, 1), (896, 12, 1), (896, 8, 2), (1536, 10, 1), (2048, 12, 4), (4096, 10, 1), (5120, 12, 1), (5120, 12, 4),
                                      (5248, 12, 4), (8192, 12, 1), (8960, 10, 1), (17408, 12, 4)])
@pytest.mark.parametrize("R", [1, 300])
def test_against_the_oracle(R, C, bits, G):
    s = synth(R, C, 4, bits, G, 1, seed=R + C + bits)
    lin, w = to_device(s), s.decode().astype(np.float64)
    for B, dtype in ((2, torch.bfloat16), (3, torch.float16), (8, torch.bfloat16), (9, torch.float16), (16, torch.bfloat16), (17, torch.float16), (32, torch.bfloat16)):
        x = rand_x(B, C, dtype, seed=B)
        y = torch.full((B, R), float("nan"), device="cuda")
        linear_small([lin], x.cuda(), y)
        # products of fp16 values are exact in fp32; C sums of them round at 2^-24 of a partial sum, in any order: below
        # sqrt(C) 2^-24 of the largest result by a wide margin
        assert rel_max_err(y.cpu().numpy(), x.half().float().numpy().astype(np.float64) @ w.T) < 1e-5, B
