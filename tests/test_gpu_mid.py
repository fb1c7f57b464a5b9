"""Products of 33 to 2048 activation rows whose codewords are gathered once per block of them: edges of the tiles of rows and activation rows, a last round
with missing units, odd numbers of rounds, K slices, stacks, several codebooks, two tiles of rows per wave, two parts of rows; and
of 3 to 256 rows with weights decoded first; and decode batches of 17 to 32."""

import ctypes

import numpy as np
import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import linear_gemm, linear_small
from tests.helpers import rand_x, rel_max_err, synth, to_device, with_infinity

pytestmark = pytest.mark.gpu

CASES = [  # rows of the stack's pieces, C, d, bits, G, T
    ((1,), 64, 8, 16, 1, 33), ((15, 17), 320, 8, 16, 1, 48), ((129,), 3584, 8, 16, 1, 49), ((513, 128), 1600, 8, 16, 2, 81),
    ((66,), 704, 8, 16, 1, 256), ((33000,), 128, 8, 16, 1, 250),
    ((1,), 32, 4, 12, 1, 80), ((127, 3, 260), 1056, 4, 12, 1, 128), ((130,), 2080, 4, 12, 4, 129), ((64, 70), 1024, 4, 12, 4, 256),
    ((33001,), 160, 4, 12, 1, 193), ((32768,), 96, 4, 12, 1, 241), ((4096,), 16384, 4, 12, 1, 257),
    ((16, 1, 130, 40, 7, 64, 33, 20), 512, 8, 16, 1, 70), ((30, 1, 17, 64, 8, 9, 130), 1024, 4, 12, 1, 40), ((24,) * 9, 512, 8, 16, 1, 90),
    # ten and twelve waves per workgroup
    ((33000,), 64, 8, 16, 1, 34), ((16500, 16501), 192, 8, 16, 1, 80), ((41500,), 64, 8, 16, 1, 65), ((33003,), 64, 8, 16, 1, 128),
    ((33001,), 96, 4, 12, 1, 50), ((41000, 30), 64, 4, 10, 1, 70), ((33000,), 64, 4, 8, 1, 33), ((33000,), 96, 4, 12, 4, 150), ((33000,), 96, 4, 12, 2, 150),
    ((257,), 576, 4, 10, 1, 192), ((40, 8), 1600, 4, 10, 2, 34), ((131,), 1536, 4, 8, 1, 129), ((36,), 64, 4, 8, 1, 255),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("stream", [True, False], ids=["tiled", "rows"])
def test_one_pass_matches_oracle(case, dtype, stream):
    rows, C, d, bits, G, T = case
    ss = [synth(R, C, d, bits, G, 1, seed=R + T) for R in rows]
    lins = [to_device(s, stream=stream and d == 4) for s in ss]
    x = rand_x(T, C, dtype, seed=T)
    ref = torch.cat([x.cuda().double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    y = torch.empty(T, sum(rows), dtype=torch.float32, device="cuda")
    linear_gemm(lins, x.cuda(), y)
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-3
    lowp = torch.empty(T, sum(rows), dtype=dtype, device="cuda")
    linear_gemm(lins, x.cuda(), lowp)
    assert torch.equal(lowp, y.to(dtype))
    assert np.isfinite(lowp.float().cpu().numpy()).all()


# rows of the stack's pieces, C, d, bits, G, T, and the cut: tiles of activation rows, tiles of weight rows, waves, K slices.  The last block of
# activation rows and the last tile of weight rows are broken, products beyond 256 rows among them.
CUTS = [
    ((1,), 32, 4, 12, 1, 33, (1, 1, 4, 1)), ((17,), 1600, 4, 10, 1, 34, (1, 1, 4, 4)), ((8218,), 32, 4, 12, 1, 33, (1, 1, 8, 1)),
    ((5383, 5), 32, 4, 12, 1, 50, (2, 1, 4, 1)), ((8229,), 96, 4, 12, 1, 66, (2, 1, 8, 1)), ((16854,), 32, 4, 12, 1, 35, (3, 1, 8, 1)),
    ((16647,), 32, 4, 12, 1, 65, (3, 1, 10, 1)), ((41028,), 32, 4, 12, 1, 33, (3, 1, 12, 1)), ((16769,), 32, 4, 12, 1, 99, (3, 2, 8, 1)),
    ((20862,), 32, 4, 12, 1, 49, (4, 1, 8, 1)), ((41153,), 32, 4, 12, 1, 53, (4, 2, 8, 1)), ((25822,), 32, 4, 12, 1, 66, (5, 1, 8, 1)),
    ((33221,), 32, 4, 12, 1, 67, (5, 1, 10, 1)), ((41558,), 32, 4, 12, 1, 70, (5, 1, 12, 1)), ((41228,), 32, 4, 12, 1, 206, (5, 2, 8, 1)),
    ((700,), 512, 4, 12, 1, 1000, (2, 1, 8, 1)), ((3584,), 1024, 4, 8, 1, 385, (3, 1, 8, 1)), ((9225,), 64, 4, 8, 1, 419, (5, 2, 8, 1)),
    ((8588,), 32, 4, 12, 4, 33, (1, 1, 8, 1)), ((16934,), 32, 4, 12, 4, 99, (3, 2, 8, 1)), ((25828,), 32, 4, 12, 4, 68, (5, 1, 8, 1)),
    ((33375,), 32, 4, 12, 4, 67, (5, 2, 8, 1)), ((33294,), 32, 4, 12, 4, 81, (8, 2, 8, 1)), ((3000, 50), 640, 4, 10, 4, 700, (3, 1, 12, 1)),
    ((1,), 64, 8, 16, 1, 33, (1, 1, 4, 1)), ((1217,), 64, 8, 16, 1, 50, (2, 1, 4, 1)), ((3,), 2112, 8, 16, 1, 250, (2, 1, 4, 5)),
    ((560, 33), 2112, 8, 16, 1, 33, (3, 1, 4, 5)), ((17153,), 64, 8, 16, 1, 34, (3, 1, 8, 1)), ((33795,), 64, 8, 16, 1, 33, (3, 1, 10, 1)),
    ((41550,), 64, 8, 16, 1, 37, (3, 1, 12, 1)), ((1091,), 1664, 8, 16, 2, 51, (4, 1, 4, 4)), ((3571,), 2112, 8, 16, 1, 49, (4, 1, 8, 5)),
    ((4587,), 64, 8, 16, 1, 67, (5, 1, 4, 1)), ((5448,), 64, 8, 16, 1, 194, (5, 1, 8, 1)), ((33034,), 64, 8, 16, 1, 51, (5, 1, 10, 1)),
    ((41105,), 64, 8, 16, 1, 49, (5, 1, 12, 1)), ((13449,), 64, 8, 16, 1, 83, (8, 1, 8, 1)), ((33589,), 64, 8, 16, 1, 84, (8, 1, 12, 1)),
    ((2254,), 3136, 8, 16, 1, 161, (12, 1, 8, 7)), ((42185,), 64, 8, 16, 2, 130, (12, 1, 12, 1)), ((4174,), 2112, 8, 16, 1, 247, (16, 1, 8, 5)),
    ((600,), 512, 8, 16, 1, 1300, (5, 1, 4, 1)), ((49522, 49522), 64, 8, 16, 1, 56, (5, 2, 8, 1)), ((50627, 50627), 64, 8, 16, 2, 90, (8, 2, 8, 1)),
    ((43505, 10876, 10876), 64, 8, 16, 1, 131, (12, 2, 8, 1)), ((43965, 10991, 10991), 64, 8, 16, 1, 195, (16, 2, 8, 1)),
    ((806,), 64, 4, 8, 1, 1766, (3, 1, 4, 1)), ((157,), 3392, 4, 8, 1, 684, (4, 1, 4, 7)), ((165,), 5248, 4, 8, 1, 1052, (5, 1, 4, 6)),
    ((1, 1, 1), 3200, 4, 10, 4, 1430, (8, 1, 8, 7)), ((58824,), 32, 4, 12, 1, 98, (8, 2, 8, 1)),
]


@pytest.mark.parametrize("case", CUTS, ids=lambda c: "x".join(map(str, c[:-1])))
@pytest.mark.parametrize("dtype,stream", [(torch.bfloat16, True), (torch.float16, False)], ids=["bf16-tiled", "f16-rows"])
def test_cuts_match_oracle(case, dtype, stream):
    rows, C, d, bits, G, T, cut = case
    ss = [synth(R, C, d, bits, G, 1, seed=R + T) for R in rows]
    lins = [to_device(s, stream=stream and d == 4) for s in ss]
    mats = _lib.matrix_array([m.descriptor(o) for m, o in zip(lins, np.cumsum([0] + list(rows)).tolist())])
    v = _lib.lib().sq_mid_variant_for_tests(mats, len(lins), T)
    kernel = _lib.lib().sq_gemm_kernel_for_tests(mats, len(lins), T, _lib.DTYPES[dtype], (ctypes.c_float * 3)())
    # (the figures of the estimates are for 256 compute units; 3: the call below runs there)
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or (tuple(v >> k & 255 for k in (0, 8, 16, 24)) == cut and kernel == 3)
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    ref = torch.cat([xd.double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    y = torch.empty(T, sum(rows), dtype=torch.float32, device="cuda")
    linear_gemm(lins, xd, y)
    # products of fp16 values are exact in fp32, whose sums of C terms round at 2^-24 of a partial sum
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-5
    lowp = torch.zeros(T, sum(rows) + 8, dtype=dtype, device="cuda")
    linear_gemm(lins, xd, lowp[:, :sum(rows)])
    assert torch.equal(lowp[:, :sum(rows)], y.to(dtype)) and not lowp[:, sum(rows):].any()


# rows of the stack's pieces, C, bits, G, T, and how many of the pieces (d = 4, up to 32 activation rows) go that way: one and two tiles of activation
# rows, the last one broken, K slices, several codebooks, more pieces than a launch takes; a pair that SiLU could be fused behind, 16 rows
DECODE_BATCHES = [
    ((4863,), 896, 8, 1, 17, 1), ((4864,), 896, 8, 1, 32, 1), ((4864,), 896, 8, 1, 16, 0), ((16546,), 832, 10, 1, 31, 1), ((15002, 9), 512, 10, 4, 24, 2),
    ((2501,), 9408, 12, 1, 17, 1), ((17000, 17001), 1600, 12, 4, 32, 2), ((9000, 9001), 2080, 12, 4, 17, 0), ((540,) * 9, 512, 8, 4, 20, 8), ((4864, 4864), 1024, 8, 1, 20, 0), ((20000,), 640, 12, 1, 18, 1),
    ((14570, 3642, 3641), 1088, 12, 1, 32, 3),
]


@pytest.mark.parametrize("case", DECODE_BATCHES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("dtype,stream", [(torch.bfloat16, True), (torch.float16, False)], ids=["bf16-tiled", "f16-rows"])
def test_decode_batches_match_oracle(case, dtype, stream):
    rows, C, bits, G, T, pieces = case
    ss = [synth(R, C, 4, bits, G, 1, seed=R + T + i) for i, R in enumerate(rows)]
    lins = [to_device(s, stream=stream) for s in ss]
    taken = _lib.lib().sq_mid_pieces_for_tests(_lib.matrix_array([m.descriptor() for m in lins]), len(lins), T)
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or taken == pieces
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    ref = torch.cat([xd.double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    y = torch.empty(T, sum(rows), dtype=torch.float32, device="cuda")
    linear_small(lins, xd, y)
    # products of fp16 values are exact in fp32, whose sums of C terms round at 2^-24 of a partial sum
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-5
    lowp = torch.zeros(T, sum(rows) + 8, dtype=dtype, device="cuda")
    linear_small(lins, xd, lowp[:, :sum(rows)])
    assert torch.equal(lowp[:, :sum(rows)], y.to(dtype)) and not lowp[:, sum(rows):].any()


@pytest.mark.parametrize("rows,C,bits,G,T", [((17000, 17001), 1600, 12, 4, 32), ((2501,), 9408, 12, 1, 17), ((540,) * 9, 512, 8, 4, 20)], ids=lambda v: str(v))
def test_decode_batches_have_the_same_sums_without_a_workspace_argument(rows, C, bits, G, T):
    lins = [to_device(synth(R, C, 4, bits, G, 1, seed=R + T + i)) for i, R in enumerate(rows)]
    mats = _lib.matrix_array([m.descriptor(o) for m, o in zip(lins, np.cumsum([0] + list(rows)).tolist())])
    x = rand_x(T, C, torch.bfloat16, seed=T).cuda()
    y, z = torch.empty(2, T, sum(rows), device="cuda")
    linear_small(lins, x, y)
    _lib.check(_lib.lib().sq_linear_small_noalloc(mats, len(lins), x.data_ptr(), _lib.SQ_BF16, C, z.data_ptr(), _lib.SQ_F32, sum(rows), T, _lib.stream_ptr(x.device)))
    assert torch.equal(z, y)


@pytest.mark.parametrize("T", [64, 500])
def test_least_workspace_is_enough_and_less_is_refused(T):
    """K slices are as many as the workspace holds; what a call refused for lack of it is refused."""
    L, R, C = _lib.lib(), 300, 4096
    s = synth(R, C, 4, 12, seed=T)
    lin, x = to_device(s), rand_x(T, C, torch.float16, seed=T).cuda()
    mats = [lin.descriptor(0)]
    ref = x.double() @ torch.from_numpy(s.decode()).cuda().double().T
    y = torch.empty(T, R, device="cuda")
    ws = torch.zeros(L.sq_workspace_bytes(_lib.matrix_array(mats), 1, T, 3), dtype=torch.uint8, device="cuda")
    # 64 rows: 8 slices of all of them; 500: the decoded matrix, an fp16 copy of x and the sums of the tile GEMM's four parts
    least = {64: 8 * T * R * 4, 500: R * C * 2 + T * C * 2 + 8 * 4 * 128 * 256 * 4}[T]
    assert least <= ws.numel()
    call = lambda n: L.sq_linear_gemm(_lib.matrix_array(mats), 1, x.data_ptr(), _lib.SQ_F16, C, y.data_ptr(), _lib.SQ_F32, R, T, ws.data_ptr(), n, _lib.stream_ptr(x.device))
    for n in (ws.numel(), least):
        y.zero_()
        assert call(n) == 0 and rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-5
    assert call(least - 4096) == _lib.SQ_EWORKSPACE


DECODED = [  # rows of the stack's pieces, C, d, bits, G, M, T: column orders, rows of broken lane units, stages past the row's end
    ((1,), 8, 8, 16, 1, 1, 33), ((129, 1, 300), 1984, 8, 16, 1, 16, 15), ((16,), 1984, 8, 16, 1, 16, 256), ((130,), 72, 8, 16, 1, 3, 5),
    ((70, 50), 1000, 4, 12, 1, 1, 48), ((50, 16), 264, 4, 10, 4, 1, 193), ((257,), 520, 4, 8, 1, 2, 128), ((40, 40, 40, 40, 7), 512, 8, 16, 1, 2, 17),
    ((33,), 9216, 8, 16, 1, 16, 3), ((12,), 200, 2, 5, 3, 1, 81), ((3584,), 776, 8, 16, 1, 1, 100),
    ((24, 1, 33, 40, 7, 64, 9, 12, 20), 520, 8, 16, 1, 3, 60),
    ((26000, 300, 29000), 1992, 8, 16, 1, 1, 70), ((57000,), 2056, 4, 8, 1, 2, 40),      # in two steps, cut inside a piece
    ((12500, 100), 2048, 8, 16, 1, 16, 129),      # past 128 rows and 24 M weights, in tiles
]


@pytest.mark.parametrize("case", DECODED, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_decoded_weights_match_oracle(case, dtype):
    rows, C, d, bits, G, M, T = case
    ss = [synth(R, C, d, bits, G, M, seed=R + T) for R in rows]
    lins = [to_device(s) for s in ss]
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    ref = torch.cat([xd.double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    y = torch.empty(T, sum(rows), dtype=torch.float32, device="cuda")
    linear_gemm(lins, xd, y)
    assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-3


def test_empty_pieces_of_a_decoded_stack():
    L, C, T = _lib.lib(), 72, 40
    lin = to_device(synth(30, C, 8, 16, seed=1))
    x = rand_x(T, C, torch.float16, seed=2).cuda()
    ref = x.double() @ torch.from_numpy(synth(30, C, 8, 16, seed=1).decode()).cuda().double().T
    for rows in ((0,), (0, 30, 0), (0, 0)):
        mats = []
        for R in rows:
            mats.append(lin.descriptor(0))
            mats[-1].R = R
        y = torch.zeros(T, 30, device="cuda")
        ws = torch.zeros(max(L.sq_workspace_bytes(_lib.matrix_array(mats), len(mats), T, 1), 256), dtype=torch.uint8, device="cuda")
        _lib.check(L.sq_linear_gemm(_lib.matrix_array(mats), len(mats), x.data_ptr(), _lib.SQ_F16, C, y.data_ptr(), _lib.SQ_F32, 30, T, ws.data_ptr(),
                                    ws.numel(), _lib.stream_ptr(x.device)))
        assert rel_max_err(y.cpu().numpy(), ref.cpu().numpy()) < 1e-3 if 30 in rows else not y.any()


@pytest.mark.parametrize("T,ld", [(40, 1 << 26), (5, 1 << 29)])
def test_decoded_weights_with_activation_rows_that_span_4_gb(T, ld):
    s = synth(70, 520, 8, 16, 1, 3, seed=T)
    lin = to_device(s, stream=False)
    x = rand_x(T, 520, torch.bfloat16, seed=T)
    big = torch.empty((T - 1) * ld + 520, dtype=torch.bfloat16, device="cuda")
    xd = big.as_strided((T, 520), (ld, 1))
    xd.copy_(x)
    y = torch.empty(T, 70, dtype=torch.float32, device="cuda")
    linear_gemm([lin], xd, y)
    assert rel_max_err(y.cpu().numpy(), x.double().numpy() @ s.decode().astype(np.float64).T) < 1e-3


@pytest.mark.parametrize("R,C,d,bits,G,M,T", [(129, 64, 8, 16, 1, 1, 33), (300, 320, 8, 16, 2, 1, 120), (40, 2112, 8, 16, 1, 1, 250), (60, 72, 8, 16, 1, 1, 5),
                                              (70, 1000, 4, 12, 1, 1, 48), (50, 1984, 8, 16, 1, 3, 100)])
def test_missing_units_meet_no_codeword(R, C, d, bits, G, M, T):
    """A last round with missing units (or, of decoded weights, missing columns) behind a row that ends in a codeword with an infinity:
    the row's results are infinite, not NaN."""
    s = with_infinity(synth(R, C, d, bits, G, M, seed=R), 5)
    x = rand_x(T, C, torch.float16, seed=T).abs() + 0.125
    y = torch.empty(T, R, dtype=torch.float32, device="cuda")
    linear_gemm([to_device(s, stream=d == 4)], x.cuda(), y)     # (the slice stream is a layout for fewer rows)
    ref = torch.from_numpy(s.decode()).cuda().double()
    assert bool(torch.isposinf(y[:, 5]).all()) and bool(torch.isinf(ref[5]).any())
    ref[5] = 0
    y[:, 5] = 0
    # exact products and fp32 sums; weights that were decoded first are rounded to fp16 with their scale, 2^-11 of each
    assert rel_max_err(y.cpu().numpy(), (x.cuda().double() @ ref.T).cpu().numpy()) < (1e-5 if C % 64 == 0 and M == 1 else 5e-4)
