"""Products of 129 to 768 activation rows whose weights are gathered on their way into LDS: every number of token and weight tiles a
workgroup takes, edges of tiles, pieces and token blocks, rounds with missing units, odd numbers of rounds, K slices, several
codebooks, results that allow no 16-byte stores."""

import ctypes

import numpy as np
import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import linear_gemm
from tests.helpers import rand_x, rel_max_err, synth, to_device, with_infinity

pytestmark = pytest.mark.gpu

# rows of the stack's pieces, C, d, bits, G, T, and the variant: token tiles, weight tiles of a wave, K slices, token blocks (None: another kernel)
CASES = [
    ((11003,), 64, 8, 16, 1, 129, (3, 2, 1, 1)), ((9000, 130, 9001), 320, 8, 16, 1, 192, (3, 3, 1, 1)), ((24600, 8), 64, 8, 16, 1, 160, (3, 4, 1, 1)),
    ((33000,), 192, 8, 16, 1, 191, (3, 5, 1, 1)), ((6001,), 192, 8, 16, 1, 200, (4, 1, 1, 1)), ((11002,), 256, 8, 16, 1, 193, (4, 2, 1, 1)),
    ((18945,), 704, 8, 16, 1, 255, (4, 3, 1, 1)), ((25000, 1), 128, 8, 16, 1, 256, (4, 4, 1, 1)), ((32000,), 64, 8, 16, 2, 250, (4, 4, 1, 1)),
    ((38402,), 320, 8, 16, 1, 210, (4, 5, 1, 1)), ((12288,), 64, 8, 16, 1, 257, (6, 2, 1, 1)), ((18433,), 576, 8, 16, 1, 383, (6, 3, 1, 1)),
    ((24577, 16), 64, 8, 16, 1, 333, (6, 4, 1, 1)), ((40960,), 64, 8, 16, 1, 384, (6, 5, 1, 1)), ((12100,), 128, 8, 16, 1, 768, (6, 3, 1, 2)),
    ((3503,), 16384, 8, 16, 1, 150, (3, 3, 6, 1)), ((54000,), 64, 8, 16, 1, 300, None), ((36001,), 64, 8, 16, 1, 385, None),
    ((10900,), 96, 4, 12, 1, 140, (3, 2, 1, 1)), ((20437,), 288, 4, 12, 1, 180, (3, 3, 1, 1)), ((31693,), 288, 4, 12, 1, 177, (3, 4, 1, 1)),
    ((29000,), 160, 4, 12, 2, 150, (3, 4, 1, 1)), ((37642,), 160, 4, 12, 1, 131, (3, 5, 1, 1)), ((13540,), 96, 4, 12, 1, 235, (4, 2, 1, 1)),
    ((18784,), 160, 4, 12, 1, 201, (4, 3, 1, 1)), ((30000, 20), 160, 4, 12, 1, 256, (4, 4, 1, 1)), ((37000,), 64, 4, 12, 1, 500, (4, 5, 1, 2)),
    ((15342,), 96, 4, 12, 1, 370, (6, 2, 1, 1)), ((19000,), 1056, 4, 12, 1, 333, (6, 3, 1, 1)), ((27919,), 96, 4, 12, 1, 328, (6, 4, 1, 1)),
    ((38001,), 96, 4, 12, 1, 290, (6, 5, 1, 1)), ((3400,), 16416, 4, 12, 1, 384, (6, 3, 7, 1)),
    ((13275,), 192, 4, 10, 1, 156, (3, 2, 1, 1)), ((18991,), 192, 4, 10, 1, 188, (3, 3, 1, 1)), ((25001,), 64, 4, 10, 1, 150, (3, 4, 1, 1)),
    ((34607,), 64, 4, 10, 1, 178, (3, 5, 1, 1)), ((12636,), 320, 4, 10, 1, 233, (4, 2, 1, 1)), ((21144,), 64, 4, 10, 1, 202, (4, 3, 1, 1)),
    ((24814,), 64, 4, 10, 1, 249, (4, 4, 1, 1)), ((33001,), 64, 4, 10, 1, 220, (4, 5, 1, 1)), ((12001,), 192, 4, 10, 4, 384, (6, 2, 1, 1)),
    ((19215,), 64, 4, 10, 1, 358, (6, 3, 1, 1)), ((26158,), 64, 4, 10, 1, 370, (6, 4, 1, 1)), ((35669,), 64, 4, 10, 1, 299, (6, 5, 1, 1)),
    ((15917,), 320, 4, 8, 1, 186, (3, 2, 1, 1)), ((22625,), 64, 4, 8, 1, 143, (3, 3, 1, 1)), ((30457,), 192, 4, 8, 1, 142, (3, 4, 1, 1)),
    ((35747,), 192, 4, 8, 1, 131, (3, 5, 1, 1)), ((13000,), 64, 4, 8, 1, 193, (4, 2, 1, 1)), ((20898,), 64, 4, 8, 1, 204, (4, 3, 1, 1)),
    ((24600,), 320, 4, 8, 2, 255, (4, 4, 1, 1)), ((35461,), 192, 4, 8, 1, 198, (4, 5, 1, 1)), ((13968,), 320, 4, 8, 1, 363, (6, 2, 1, 1)),
    ((22301,), 320, 4, 8, 1, 259, (6, 3, 1, 1)), ((30353,), 192, 4, 8, 1, 349, (6, 4, 1, 1)), ((18500, 33), 1088, 4, 8, 1, 640, (6, 5, 1, 2)),
]


def _variant(lins, T):
    v = _lib.lib().sq_fused_variant_for_tests(_lib.matrix_array([m.descriptor() for m in lins]), len(lins), T)
    return tuple(v >> k & 255 for k in (0, 8, 16, 24)) if v else None


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:-1])))
@pytest.mark.parametrize("dtype,stream", [(torch.bfloat16, True), (torch.float16, False)], ids=["bf16-tiled", "f16-rows"])
def test_matches_oracle(case, dtype, stream):
    rows, C, d, bits, G, T, variant = case
    ss = [synth(R, C, d, bits, G, 1, seed=R + T) for R in rows]
    lins = [to_device(s, stream=stream and d == 4) for s in ss]
    # (the figures of the plan are for 256 compute units)
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or _variant(lins, T) == variant
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    ref = torch.cat([xd.double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    y = torch.empty(T, sum(rows), dtype=torch.float32, device="cuda")
    linear_gemm(lins, xd, y)
    # products of fp16 values are exact in fp32, whose sums of C terms round at 2^-24 of a partial sum: below sqrt(C) 2^-24 of the largest
    # result by a wide margin.  The other kernels round the decoded weights to fp16, 2^-11 of each.
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < (1e-5 if variant else 1e-3)
    lowp = torch.zeros(T, sum(rows) + 8, dtype=dtype, device="cuda")
    linear_gemm(lins, xd, lowp[:, :sum(rows)])
    assert torch.equal(lowp[:, :sum(rows)], y.to(dtype)) and not lowp[:, sum(rows):].any()
    assert np.isfinite(lowp.float().cpu().numpy()).all()


@pytest.mark.parametrize("R,C,d,bits,G,T", [(11003, 64, 8, 16, 1, 129), (24577, 320, 8, 16, 1, 333), (12100, 704, 8, 16, 1, 700), (10900, 96, 4, 12, 1, 140),
                                            (30000, 160, 4, 12, 2, 150), (12001, 192, 4, 10, 4, 384), (18500, 1088, 4, 8, 1, 640)])
def test_missing_units_meet_no_codeword(R, C, d, bits, G, T):
    """A last round with missing units, behind a row that ends in a codeword with an infinity: the row's results are infinite, not NaN."""
    s = with_infinity(synth(R, C, d, bits, G, 1, seed=R), 5)
    lin, x = to_device(s), rand_x(T, C, torch.float16, seed=T).abs() + 0.125
    y = torch.empty(T, R, dtype=torch.float32, device="cuda")
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or _variant([lin], T) is not None
    linear_gemm([lin], x.cuda(), y)
    ref = torch.from_numpy(s.decode()).cuda().double()
    assert bool(torch.isposinf(y[:, 5]).all()) and bool(torch.isinf(ref[5]).any())
    ref[5] = 0
    y[:, 5] = 0
    assert rel_max_err(y.cpu().numpy(), (x.cuda().double() @ ref.T).cpu().numpy()) < 1e-5       # (exact products, fp32 sums)


# products that other kernels are the faster ones for, and the kernel that takes them (3: small products, 6 and 7: decode and tiles)
GIVEN_UP = [(10843, 512, 4, 10, 263, (6, 1), 3), (10527, 2432, 4, 8, 578, (6, 2), 6), (10538, 768, 8, 16, 583, (6, 2), 6), (10858, 2304, 8, 16, 387, (4, 2), 7)]


@pytest.mark.parametrize("R,C,d,bits,T,cut,kernel", GIVEN_UP)
def test_runs_where_the_workspace_lets_no_other_in(R, C, d, bits, T, cut, kernel):
    """With room for no more than the activations in fragment order a product still runs here; with less it is refused."""
    L = _lib.lib()
    s = synth(R, C, d, bits, seed=R)
    lin, x = to_device(s, stream=False), rand_x(T, C, torch.float16, seed=T).cuda()
    mats = _lib.matrix_array([lin.descriptor(0)])
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or L.sq_gemm_kernel_for_tests(mats, 1, T, _lib.SQ_BF16, (ctypes.c_float * 3)()) == kernel
    ref = x.double() @ torch.from_numpy(s.decode()).cuda().double().T
    need = cut[1] * 64 * cut[0] * ((C + 255) // 256 * 256) * 2                     # blocks of tokens, 64 tokens per `cut[0]`, whole rounds of 256 columns
    ws, y = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda"), torch.empty(T, R, device="cuda")
    call = lambda n: L.sq_linear_gemm(mats, 1, x.data_ptr(), _lib.SQ_F16, C, y.data_ptr(), _lib.SQ_F32, R, T, ws.data_ptr(), n, _lib.stream_ptr(x.device))
    assert call(need) == 0 and rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-5 and bool((ws[need:] == 0x5A).all())      # (as above)
    assert call(need - 256) == _lib.SQ_EWORKSPACE


def test_runs_where_x_spans_more_than_the_others_address():
    R, C, T, ld = 11028, 512, 134, 1 << 24                                         # 4.5 GB from the first row of x to the last
    s = synth(R, C, 4, 12, seed=R)
    lin = to_device(s)
    x = torch.empty(T, ld, dtype=torch.float16, device="cuda")[:, :C]
    x.copy_(rand_x(T, C, torch.float16, seed=T))
    y = torch.empty(T, R, device="cuda")
    linear_gemm([lin], x, y)
    ref = x.double() @ torch.from_numpy(s.decode()).cuda().double().T
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-5
