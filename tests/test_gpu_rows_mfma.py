"""The matrix-core decode kernel with its codebooks in LDS, at the splits of a row over waves and workgroups that its plan makes: one
wave and sixteen, short and split rows, idle rounds in the last wave, room for 8 tokens at a time only, two token tiles."""

import numpy as np
import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import _Workspace, linear_gemm, linear_small
from oracle import sq_oracle as O
from tests.helpers import rand_x, rel_max_err, synth, to_device, with_infinity

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


@pytest.mark.parametrize("C,bits,G", [(5760, 12, 4), (6208, 12, 1), (6912, 12, 4), (7168, 8, 1), (7680, 10, 4), (8192, 12, 2), (8192, 10, 1), (8192, 8, 1)])
@pytest.mark.parametrize("rows", [(20001,), (50, 17, 300)])
def test_rows_that_one_launch_takes_whole(rows, C, bits, G):
    """Stacks and tall matrices, and any of these where the workspace has no room for partial sums (none at all here)."""
    L, dev = _lib.lib(), torch.device("cuda", torch.cuda.current_device())
    ss = [synth(R, C, 4, bits, G, 1, seed=R + C) for R in rows]
    lins = [to_device(s) for s in ss]
    w = torch.cat([torch.from_numpy(s.decode()).cuda().double() for s in ss])
    offs = [sum(rows[:i]) for i in range(len(rows))]
    for B, dtype in ((2, torch.bfloat16), (5, torch.float16), (8, torch.bfloat16), (9, torch.float16), (16, torch.bfloat16)):
        x = rand_x(B, C, dtype, seed=B).cuda()
        want = (x.half().double() @ w.T).cpu().numpy()
        y = torch.full((B, sum(rows)), float("nan"), device="cuda")
        linear_small(lins, x, y)
        assert rel_max_err(y.cpu().numpy(), want) < 1e-5, B         # (see above)
        for off, lin in ((offs, lins), ([0], lins[:1])):
            mats = _lib.matrix_array([m.descriptor(o) for m, o in zip(lin, off)])
            n = sum(m.R for m in lin)
            y.fill_(float("nan"))
            _lib.check(L.sq_linear_small(mats, len(lin), x.data_ptr(), _lib.DTYPES[dtype], C, y.data_ptr(), _lib.SQ_F32, sum(rows), B, None, 0,
                                         _lib.stream_ptr(dev)))
            assert rel_max_err(y[:, :n].cpu().numpy(), want[:, :n]) < 1e-5 and bool(y[:, n:].isnan().all()), B


@pytest.mark.parametrize("rows", [(40,), (37, 64, 21), (33, 40)])
@pytest.mark.parametrize("C,bits", [(18944, 12), (66560, 12), (98304, 8)])       # 5 slices, and more than eight
def test_sums_of_slices(rows, C, bits):
    """Rows in quads and not, pieces behind pieces of odd rows (whose results then begin anywhere), every result type."""
    ss = [synth(R, C, 4, bits, 1, 1, seed=R + bits) for R in rows]
    lins, w = [to_device(s) for s in ss], np.concatenate([s.decode().astype(np.float64) for s in ss])
    for dtype, tol in ((torch.float32, 1e-5), (torch.float16, 2.0 ** -11 + 1e-5), (torch.bfloat16, 2.0 ** -8 + 1e-5)):      # (the first as above)
        x = rand_x(3, C, torch.float16 if dtype == torch.float32 else dtype, seed=C)
        want = x.half().float().numpy().astype(np.float64) @ w.T
        y = torch.full((3, sum(rows)), float("nan"), dtype=dtype, device="cuda")
        linear_small(lins, x.cuda(), y)
        assert rel_max_err(y.float().cpu().numpy(), want) < tol, dtype


@pytest.mark.parametrize("rows,C,bits,G,B", [((300,), 8192, 12, 1, 8), ((300,), 6912, 12, 4, 16), ((40, 300), 7168, 8, 1, 2)])
@pytest.mark.parametrize("native", [True, False], ids=["native", "python"])
def test_products_that_need_no_sums_share_nothing(rows, C, bits, G, B, native, monkeypatch):
    """The partial sums of rows that one launch could take whole leave the shared workspace alone (two streams may run them at once),
    eagerly and in a graph, each replay the same."""
    if not native:
        monkeypatch.setattr(_lib.native(), "linear", lambda *a: 1)
    ss = [synth(R, C, 4, bits, G, 1, seed=R + C) for R in rows]
    lins = [to_device(s) for s in ss]
    x = rand_x(B, C, torch.bfloat16, seed=B).cuda()
    mats = _lib.matrix_array([m.descriptor() for m in lins])
    shared = _Workspace.get(_lib.lib().sq_workspace_bytes(mats, len(lins), B, 0), x.device)[_lib.WS_HEADER:]
    shared.fill_(0x5A)
    y = torch.empty(B, sum(rows), device="cuda")
    linear_small(lins, x, y)
    want = np.concatenate([x.cpu().half().double().numpy() @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.cpu().numpy(), want) < 1e-5 and bool((shared == 0x5A).all())
    first = y.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        linear_small(lins, x, y)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, first) and bool((shared == 0x5A).all())


@pytest.mark.parametrize("C,bits,G", [(8, 12, 1), (40, 10, 1), (72, 8, 1), (1360, 10, 4), (2056, 12, 1), (2080, 8, 4), (2928, 10, 1), (5624, 12, 4), (6168, 8, 1),
                                      (8968, 12, 1), (17416, 10, 1)])
@pytest.mark.parametrize("rows", [(1,), (300, 17)])
def test_rows_that_end_within_a_unit(rows, C, bits, G):
    """Their tile-major copy is filled up to whole units, and what lies behind a row stays out of its results: the columns of x (NaN here)
    and the codewords of the filling (an infinity that no other tag names)."""
    ss = [synth(R, C, 4, bits, G, 1, seed=R + C) for R in rows]
    for s in ss:
        s.tags[:] = np.maximum(s.tags, 1)
        s.words[:] = O.pack_bits(s.tags, bits)
        s.table[:: s.K] = np.inf
    lins = [to_device(s) for s in ss]
    assert all(m.stream_tiled for m in lins)
    w = torch.cat([torch.from_numpy(s.decode()).cuda().double() for s in ss])
    for B, dtype in ((1, torch.bfloat16), (2, torch.float16), (8, torch.bfloat16), (16, torch.float16), (17, torch.bfloat16), (32, torch.float16),
                     (33, torch.bfloat16), (77, torch.float16), (200, torch.bfloat16), (260, torch.float16)):
        x = torch.full((B, C + 64), float("nan"), dtype=dtype, device="cuda")
        x[:, :C] = rand_x(B, C, dtype, seed=B).cuda()
        x = x[:, :C]
        y = torch.full((B, sum(rows)), float("nan"), device="cuda")
        (linear_small if B <= 32 else linear_gemm)(lins, x, y)
        assert rel_max_err(y.cpu().numpy(), (x.half().double() @ w.T).cpu().numpy()) < 1e-5, B      # (see above)


def test_infinity_at_the_end_of_a_broken_row():
    s = with_infinity(synth(70, 2056, 4, 12, seed=1), 5)
    for B in (1, 8, 32):
        x = rand_x(B, 2056, torch.float16, seed=B).abs() + 0.125
        y = torch.empty(B, 70, device="cuda")
        linear_small([to_device(s)], x.cuda(), y)
        assert bool(torch.isposinf(y[:, 5]).all()) and bool(y[:, :5].isfinite().all()) and bool(y[:, 6:].isfinite().all())


@pytest.mark.parametrize("C,B", [(2056, 16), (17416, 8), (17416, 40)])
def test_rows_that_end_within_a_unit_without_a_workspace(C, B):
    """What ran without one before such rows had a copy still does."""
    L, dev = _lib.lib(), torch.device("cuda", torch.cuda.current_device())
    s = synth(70, C, 4, 12, seed=C)
    lin = to_device(s)
    x = rand_x(B, C, torch.float16, seed=B).cuda()
    y = torch.full((B, 70), float("nan"), device="cuda")
    call = L.sq_linear_small if B <= 32 else L.sq_linear_gemm
    _lib.check(call(_lib.matrix_array([lin.descriptor()]), 1, x.data_ptr(), _lib.SQ_F16, C, y.data_ptr(), _lib.SQ_F32, 70, B, None, 0, _lib.stream_ptr(dev)))
    assert rel_max_err(y.cpu().numpy(), x.cpu().double().numpy() @ s.decode().astype(np.float64).T) < 1e-5


@pytest.mark.parametrize("d,bits,C,G", [(8, 16, 2080, 1), (8, 16, 5000, 1), (8, 14, 1024, 1), (4, 14, 512, 1), (4, 12, 2056, 8), (8, 5, 264, 1)])
@pytest.mark.parametrize("room", [True, False])
def test_formats_of_the_vector_kernels(d, bits, C, G, room):
    """From three rows their weights are decoded first, where the workspace has room."""
    L, dev = _lib.lib(), torch.device("cuda", torch.cuda.current_device())
    ss = [synth(R, C, d, bits, G, 1, seed=R) for R in (130, 9)]
    lins = [to_device(s, stream=False) for s in ss]
    w = np.concatenate([s.decode() for s in ss]).astype(np.float64)
    for B in (2, 3, 9, 32):
        x = rand_x(B, C, torch.bfloat16, seed=B).cuda()
        y = torch.full((B, 139), float("nan"), device="cuda")
        if room:
            linear_small(lins, x, y)
        else:
            mats = _lib.matrix_array([lins[0].descriptor(0), lins[1].descriptor(130)])
            _lib.check(L.sq_linear_small(mats, 2, x.data_ptr(), _lib.SQ_BF16, C, y.data_ptr(), _lib.SQ_F32, 139, B, None, 0, _lib.stream_ptr(dev)))
        assert rel_max_err(y.cpu().numpy(), x.half().double().cpu().numpy() @ w.T) < 1e-5, B


@pytest.mark.parametrize("d,bits", [(8, 16), (4, 12)])
@pytest.mark.parametrize("stream", [True, False])
@pytest.mark.parametrize("noalloc", [True, False])
def test_mixed_stacks(d, bits, stream, noalloc):
    """Pieces that are decoded first beside pieces whose tags are read: each runs as it does alone."""
    L, C = _lib.lib(), 1024
    formats = [(700, d, bits), (40, 8, 14), (33, 4, 14), (300, d, bits), (17, 8, 5)]
    ss = [synth(R, C, dd, b, 1, 1, seed=R) for R, dd, b in formats]
    lins = [to_device(s, stream=stream) for s in ss]
    R = sum(f[0] for f in formats)
    w = np.concatenate([s.decode() for s in ss]).astype(np.float64)
    for B in (2, 3, 9, 32):
        x = rand_x(B, C, torch.bfloat16, seed=B).cuda()
        y = torch.full((B, R), float("nan"), device="cuda")
        if noalloc:
            offs = np.cumsum([0] + [f[0] for f in formats])
            mats = _lib.matrix_array([lin.descriptor(int(o)) for lin, o in zip(lins, offs)])
            _lib.check(L.sq_linear_small_noalloc(mats, len(lins), x.data_ptr(), _lib.SQ_BF16, C, y.data_ptr(), _lib.SQ_F32, R, B, _lib.stream_ptr(x.device)))
        else:
            linear_small(lins, x, y)
        assert rel_max_err(y.cpu().numpy(), x.half().double().cpu().numpy() @ w.T) < 1e-5, B
        for i in (0, 3):
            o = sum(f[0] for f in formats[:i])
            alone = torch.empty(B, formats[i][0], device="cuda")
            linear_small([lins[i]], x, alone)
            assert torch.equal(y[:, o:o + formats[i][0]], alone), (B, i)


def _wide_activations(B, C, seed):
    """bf16 rows that fp16 does not hold: far below its normal range, far beyond its largest value, a few of those among ordinary ones, at
    the row's end alone, one ordinary value among tiny ones, all zero."""
    x = rand_x(B, C, torch.bfloat16, seed=seed).float()
    for b in range(B):
        kind = b % 8
        if kind == 1: x[b] *= 1e-7
        if kind == 2: x[b, 5], x[b, C // 2], x[b, C - 9] = 1e5, -3e6, 70000.0
        if kind == 3: x[b] *= 1e28
        if kind == 4: x[b] = 0.0
        if kind == 5: x[b] = 0.0; x[b, C - 1] = 2e5
        if kind == 6: x[b] *= 2.0 ** -20; x[b, 11] = 1.0
        if kind == 7: x[b] *= 3e-13; x[b, C // 3] = 4e-12
    return x.to(torch.bfloat16)


def _check_wide_activations(lins, w, C, rows):
    for B in rows:
        x = _wide_activations(B, C, seed=B)
        y = torch.full((B, w.shape[0]), float("nan"), device="cuda")
        linear_small(lins, x.cuda(), y)
        y, ref = y.cpu().double().numpy(), x.double().numpy() @ w.T
        # (sums of products that are exact in 32 bits or below 2^-24 of the largest one: as for ordinary activations)
        for b in range(B):
            assert np.abs(y[b] - ref[b]).max() <= 1e-5 * np.abs(ref[b]).max(), (B, b)
        # what is not finite, beside finite values that fp16 does not hold
        x[0, 3], x[0, 9] = float("inf"), 1e6
        x[B - 1, C - 2] = float("nan")
        y = torch.zeros(B, w.shape[0], device="cuda")
        linear_small(lins, x.cuda(), y)
        with np.errstate(invalid="ignore"):
            ref = x.double().numpy() @ w.T
        y = y.cpu().double().numpy()
        for b in {0, B - 1}:
            assert np.array_equal(np.isnan(y[b]), np.isnan(ref[b])) and np.array_equal(np.isposinf(y[b]), np.isposinf(ref[b])) and \
                np.array_equal(np.isneginf(y[b]), np.isneginf(ref[b])), (B, b)


@pytest.mark.parametrize("rows,C,bits,G", [((100, 7), 2056, 12, 1), ((70,), 904, 8, 1), ((70,), 1000, 10, 4), ((33,), 9224, 12, 1), ((33,), 5672, 12, 4), ((20,), 40, 12, 1)])
def test_activations_beyond_fp16_of_broken_rows(rows, C, bits, G):
    """Rows that end within a lane unit: bf16 activations keep their range and their bits."""
    ss = [synth(R, C, 4, bits, G, 1, seed=R) for R in rows]
    lins = [to_device(s) for s in ss]
    _check_wide_activations(lins, np.concatenate([s.decode() for s in ss]).astype(np.float64), C, (1, 2, 7, 9, 16, 17, 32))


@pytest.mark.parametrize("rows,C,d,bits,G", [((700, 9), 2080, 8, 16, 1), ((5000,), 5000, 8, 16, 1), ((900,), 1024, 8, 14, 1), ((2000,), 1024, 4, 14, 1), ((600,), 2056, 4, 12, 8),
                                             ((4000,), 264, 8, 5, 1)])
def test_activations_beyond_fp16_of_vector_formats(rows, C, d, bits, G):
    """Formats without a matrix-core kernel, decoded first or not: bf16 activations keep their range and their bits."""
    ss = [synth(R, C, d, bits, G, 1, seed=R) for R in rows]
    lins = [to_device(s, stream=False) for s in ss]
    _check_wide_activations(lins, np.concatenate([s.decode() for s in ss]).astype(np.float64), C, (1, 3, 8, 16, 17, 32))
