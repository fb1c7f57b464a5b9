"""Products of 129 to 768 activation rows whose weights are gathered on their way into LDS: every number of token and weight tiles a
workgroup takes, edges of tiles, pieces and token blocks, rounds with missing units, odd numbers of rounds, K slices, several
codebooks, results that allow no 16-byte stores."""

import numpy as np
import pytest
import torch

from quantexperiments_amd.kernels import linear_gemm
from tests.helpers import rand_x, rel_max_err, synth, to_device, with_infinity

pytestmark = pytest.mark.gpu

CASES = [  # rows of the stack's pieces, C, d, bits, G, T
    ((11003,), 64, 8, 16, 1, 129), ((9000, 130, 9001), 320, 8, 16, 1, 192), ((24600, 8), 64, 8, 16, 1, 160), ((33000,), 192, 8, 16, 1, 191),
    ((6001,), 192, 8, 16, 1, 200), ((11002,), 256, 8, 16, 1, 193), ((18945,), 704, 8, 16, 1, 255), ((25000, 1), 128, 8, 16, 1, 256), ((32000,), 64, 8, 16, 2, 250),
    ((12288,), 64, 8, 16, 1, 257), ((18433,), 576, 8, 16, 1, 383), ((24577, 16), 64, 8, 16, 1, 333), ((40960,), 64, 8, 16, 1, 384), ((54000,), 64, 8, 16, 1, 300),
    ((36001,), 64, 8, 16, 1, 385), ((12100,), 128, 8, 16, 1, 768), ((3503,), 16384, 8, 16, 1, 150),
    ((10900,), 96, 4, 12, 1, 140), ((30000, 20), 160, 4, 12, 1, 256), ((19000,), 1056, 4, 12, 1, 333), ((37000,), 64, 4, 12, 1, 500), ((3400,), 16416, 4, 12, 1, 384),
    ((12001,), 192, 4, 10, 4, 384), ((25001,), 64, 4, 10, 1, 150), ((33001,), 64, 4, 10, 1, 220), ((13000,), 64, 4, 8, 1, 193), ((24600,), 320, 4, 8, 2, 255),
    ((18500, 33), 1088, 4, 8, 1, 640),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("dtype,stream", [(torch.bfloat16, True), (torch.float16, False)], ids=["bf16-tiled", "f16-rows"])
def test_matches_oracle(case, dtype, stream):
    rows, C, d, bits, G, T = case
    ss = [synth(R, C, d, bits, G, 1, seed=R + T) for R in rows]
    lins = [to_device(s, stream=stream and d == 4) for s in ss]
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    ref = torch.cat([xd.double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    y = torch.empty(T, sum(rows), dtype=torch.float32, device="cuda")
    linear_gemm(lins, xd, y)
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-3
    lowp = torch.zeros(T, sum(rows) + 8, dtype=dtype, device="cuda")
    linear_gemm(lins, xd, lowp[:, :sum(rows)])
    assert torch.equal(lowp[:, :sum(rows)], y.to(dtype)) and not lowp[:, sum(rows):].any()
    assert np.isfinite(lowp.float().cpu().numpy()).all()


@pytest.mark.parametrize("R,C,d,bits,G,T", [(11003, 64, 8, 16, 1, 129), (24577, 320, 8, 16, 1, 333), (12100, 704, 8, 16, 1, 700), (10900, 96, 4, 12, 1, 140),
                                            (30000, 160, 4, 12, 2, 150), (12001, 192, 4, 10, 4, 384), (18500, 1088, 4, 8, 1, 640)])
def test_missing_units_meet_no_codeword(R, C, d, bits, G, T):
    """A last round with missing units, behind a row that ends in a codeword with an infinity: the row's results are infinite, not NaN."""
    s = with_infinity(synth(R, C, d, bits, G, 1, seed=R), 5)
    x = rand_x(T, C, torch.float16, seed=T).abs() + 0.125
    y = torch.empty(T, R, dtype=torch.float32, device="cuda")
    linear_gemm([to_device(s)], x.cuda(), y)
    ref = torch.from_numpy(s.decode()).cuda().double()
    assert bool(torch.isposinf(y[:, 5]).all()) and bool(torch.isinf(ref[5]).any())
    ref[5] = 0
    y[:, 5] = 0
    assert rel_max_err(y.cpu().numpy(), (x.cuda().double() @ ref.T).cpu().numpy()) < 1e-5       # (exact products, fp32 sums)
