"""The product that holds a slice of a large codebook in LDS and sieves the tags through it, where it can go wrong: rows that end within
tiles and quads, tiles past the last row, units past a row's end, K slices, several pieces, and activations or codewords that are not
finite; its route by the workspace it asks for."""

import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import linear_small
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu

# 2, 3, 4 and 5 tiles a wave, one to eight K slices, rounds of 4, 2, 1 and 3 units at the end; the rows beyond which the gathers from L2 run
SHAPES = [((14351,), 4160, 16), ((8100,), 9216, 16), ((2047,), 19008, 16), ((7901, 3000), 5184, 9), ((29001,), 4160, 16), ((36000,), 2112, 9), ((16001, 16, 2050), 4288, 16)]


def _pieces(rows, C):
    ss = [synth(R, C, 8, 16, 1, 1, seed=R + C) for R in rows]
    lins = [to_device(s, stream=False) for s in ss]
    return lins, torch.cat([lin.dense(torch.float32).double() for lin in lins])


def _call(lins, x, y, ws):
    mats = _lib.matrix_array([m.descriptor(o) for m, o in zip(lins, torch.tensor([0] + [m.R for m in lins]).cumsum(0).tolist())])
    _lib.check(_lib.lib().sq_linear_small(mats, len(lins), x.data_ptr(), _lib.DTYPES[x.dtype], x.stride(0), y.data_ptr(), _lib.DTYPES[y.dtype], y.stride(0),
                                          x.shape[0], None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(), _lib.stream_ptr(x.device)))


@pytest.mark.parametrize("rows,C,most", SHAPES)
def test_against_float64(rows, C, most):
    lins, w = _pieces(rows, C)
    mats = _lib.matrix_array([m.descriptor(0) for m in lins])
    for B, dtype, out in ((1, torch.bfloat16, torch.float32), (5, torch.float16, torch.float16), (9, torch.bfloat16, torch.bfloat16), (most, torch.float16, torch.float32)):
        # the eight slices' sums are what the gathers from L2 have no use for: this many bytes say which kernel runs
        assert _lib.lib().sq_workspace_bytes(mats, len(lins), B, 2) >= 32 * B * sum(rows)
        x = rand_x(B, C, dtype, seed=B).cuda()
        y = torch.full((B, sum(rows)), float("nan"), dtype=out, device="cuda")
        linear_small(lins, x, y)
        # C sums of exact products round at 2^-24 of a partial sum each, in any order: below sqrt(C) 2^-24 of the largest result
        # by a wide margin; then the result's own type
        tol = {torch.float32: 1e-5, torch.float16: 2.0 ** -11 + 1e-5, torch.bfloat16: 2.0 ** -8 + 1e-5}[out]
        assert rel_max_err(y.float().cpu().numpy(), (x.half().double() @ w.T).cpu().numpy()) < tol, B


def test_without_the_room_the_gathers_run():
    lins, w = _pieces((14351,), 4160)
    mats = _lib.matrix_array([lins[0].descriptor(0)])
    x = rand_x(9, 4160, torch.bfloat16, seed=1).cuda()
    least = _lib.lib().sq_workspace_bytes(mats, 1, 9, 4 | 2)
    assert least < 32 * 9 * 14351
    y = torch.empty(9, 14351, device="cuda")
    _call(lins, x, y, torch.empty(least, dtype=torch.uint8, device="cuda") if least else None)
    assert rel_max_err(y.cpu().numpy(), (x.half().double() @ w.T).cpu().numpy()) < 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activations_that_are_not_finite(dtype):
    """Infinite where the product is, NaN where it is, and the other rows as ever."""
    lins, w = _pieces((14351,), 4160)
    x = rand_x(6, 4160, dtype, seed=2)
    x[1, 5] = float("inf")
    x[2, 4159] = float("-inf")
    x[3, 700] = float("nan")
    if dtype == torch.bfloat16:
        x[4, 64] = 3e38                      # beyond fp16: infinite there
    x = x.cuda()
    y = torch.empty(6, 14351, device="cuda")
    linear_small(lins, x, y)
    want = x.half().double() @ w.T
    for t in range(6):
        assert torch.equal(torch.isnan(y[t]), torch.isnan(want[t])) and torch.equal(y[t] == float("inf"), want[t] == float("inf")) \
            and torch.equal(y[t] == float("-inf"), want[t] == float("-inf")), t
    assert rel_max_err(y[[0, 5]].cpu().numpy(), want[[0, 5]].cpu().numpy()) < 1e-5


def test_a_codeword_that_is_not_finite():
    """Every codeword that a row does not name leaves it alone, also past the row's end (4160 columns: a round of one unit)."""
    s = synth(14351, 4160, 8, 16, 1, 1, seed=7)
    s.table[int(s.tags[3, 11])] = float("inf")
    s.table[65535] = float("nan")
    s.table[0] = float("nan")
    lin = to_device(s, stream=False)
    w = lin.dense(torch.float32).double()
    x = rand_x(9, 4160, torch.float16, seed=3).cuda()
    y = torch.empty(9, 14351, device="cuda")
    linear_small([lin], x, y)
    want = x.double() @ w.T
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(y), ok)
    assert ((y - want).abs()[ok] < 1e-5 * want[ok].abs().max()).all()


@pytest.mark.parametrize("rows,C,T", [((18944, 18944), 3584, 16), ((18945, 3, 18946), 3584, 14), ((36000,), 3648, 16), ((60001,), 4160, 13)])
def test_sums_that_do_not_fit_at_once(rows, C, T):
    """Rows a part at a time, in the workspace there is: the bits of the whole product, through the entry point that has 16 MB behind its
    header as well."""
    lins, w = _pieces(rows, C)
    mats = _lib.matrix_array([m.descriptor(sum(rows[:i])) for i, m in enumerate(lins)])
    room = 16 << 20
    assert _lib.lib().sq_workspace_bytes(mats, len(lins), T, 2) > room
    x = rand_x(T, C, torch.bfloat16, seed=T)
    x[2, 5] = float("inf")
    x = x.cuda()
    y, z = (torch.full((T, sum(rows)), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    linear_small(lins, x, y)
    _lib.check(_lib.lib().sq_linear_small_noalloc(mats, len(lins), x.data_ptr(), _lib.SQ_BF16, C, z.data_ptr(), _lib.SQ_BF16, sum(rows), T, _lib.stream_ptr(x.device)))
    assert torch.equal(y.view(torch.int16), z.view(torch.int16))
    z.fill_(float("nan"))
    _call(lins, x, z, torch.empty(room, dtype=torch.uint8, device="cuda"))
    assert torch.equal(y.view(torch.int16), z.view(torch.int16))
    ok = [t for t in range(T) if t != 2]
    assert rel_max_err(y[ok].float().cpu().numpy(), (x[ok].half().double() @ w.T).cpu().numpy()) < 2.0 ** -8 + 1e-5
