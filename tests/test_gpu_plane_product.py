"""The product that looks up a column of a large codebook at a time: every number of token tiles and of weight tiles a wave takes, one column a
workgroup and two, rows and chunks that end within tiles, pairs of rows and steps, waves and workgroups without a tile, stacks, rounds, codewords and
activations that are not finite, and the row counts and shapes that take it."""

import ctypes

import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import linear_small
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu

_p, _i64 = ctypes.c_void_p, ctypes.c_int64


def _mats(lins):
    return _lib.matrix_array([m.descriptor(o) for m, o in zip(lins, torch.tensor([0] + [m.R for m in lins]).cumsum(0).tolist())])


def _call(lins, x, y):
    f = _lib.lib().sq_plane_product_for_tests
    f.restype = _i64
    args = (_mats(lins), len(lins), _p(x.data_ptr()), _lib.DTYPES[x.dtype], _i64(x.stride(0)), _p(y.data_ptr()), _lib.DTYPES[y.dtype], _i64(y.stride(0)), x.shape[0])
    need = f(*args, _p(None), _p(None))
    assert need > 0
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    rc = f(*args, _p(ws.data_ptr()), _p(_lib.stream_ptr(x.device)))
    torch.cuda.synchronize()
    assert rc == 0 and bool((ws[need:] == 0x5A).all())


# rows of the stack's pieces, C, T.  The chip's 256 CUs are 32 parts of the rows with one column a workgroup, of 8 waves each: 1 to 5 tiles a wave are
# up to 4096, 8192, .. 20480 rows, more are rounds; with two columns twice that
SHAPES = [((1,), 64, 17), ((15, 1, 17), 576, 33), ((4097,), 512, 32), ((8200, 31), 1088, 48), ((12300,), 704, 64), ((16500, 3), 320, 80), ((20500,), 1024, 31),
          ((24001,), 2112, 24), ((37001,), 960, 47), ((18944, 18945), 448, 63), ((30002,), 1600, 79), ((9001,), 3584, 96), ((33000,), 512, 95), ((2050,), 9216, 112), ((7000,), 5056, 111),
          ((14002, 130), 640, 127), ((4000, 1000, 999), 5056, 128), ((26000,), 128, 128), ((3584,), 18944, 40), ((64,) * 8, 1984, 20)]


@pytest.mark.parametrize("rows,C,T", SHAPES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_against_float64(rows, C, T, dtype):
    ss = [synth(R, C, 8, 16, 1, 1, seed=R + C) for R in rows]
    lins = [to_device(s, stream=False) for s in ss]
    w = torch.cat([lin.dense(torch.float32).double() for lin in lins])
    x = torch.full((T, C + 8), float("nan"), dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    y = torch.full((T, sum(rows) + 3), 7.0, dtype=torch.float32, device="cuda")
    _call(lins, xd, y[:, :sum(rows)])
    # C sums of exact products round at 2^-24 of a partial sum each, in any order: below sqrt(C) 2^-24 of the largest result by a wide margin
    assert rel_max_err(y[:, :sum(rows)].cpu().numpy(), (xd.double() @ w.T).cpu().numpy()) < 1e-5 and bool((y[:, sum(rows):] == 7).all())


def test_not_finite():
    """A codeword that is not finite touches the rows that name it, also past a row's end (a last pair of 8 chunks); activations their own row."""
    s = synth(1500, 4160, 8, 16, 1, 1, seed=7)
    s.table[int(s.tags[3, 11])] = float("inf")
    s.table[65535] = float("nan")
    s.table[0] = float("nan")
    lin = to_device(s, stream=False)
    x = rand_x(18, 4160, torch.float16, seed=3)
    x[2, 5] = float("inf")
    x[17, 4159] = float("nan")
    x = x.cuda()
    y = torch.empty(18, 1500, device="cuda")
    _call([lin], x, y)
    want = x.double() @ lin.dense(torch.float32).double().T
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(y), ok) and ((y - want).abs()[ok] < 1e-5 * want[ok].abs().max()).all()


@pytest.mark.parametrize("R,C,T", [(18944, 3584, 24), (18944, 3584, 64), (3584, 18944, 77), (14336, 5120, 100)])
def test_large_products_take_it(R, C, T):
    lin = to_device(synth(R, C, 8, 16, 1, 1, seed=5), stream=False)
    w = lin.dense(torch.float32).double()
    x = rand_x(T, C, torch.bfloat16, seed=1).cuda()
    want = torch.empty(T, R, dtype=torch.bfloat16, device="cuda")
    _call([lin], x, want)
    y = torch.empty_like(want)
    if T <= _lib.SMALL_BMAX:
        linear_small([lin], x, y)
    else:
        from quantexperiments_amd.kernels import linear_gemm
        linear_gemm([lin], x, y)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    assert rel_max_err(y.float().cpu().numpy(), (x.half().double() @ w.T).cpu().numpy()) < 2.0 ** -8 + 1e-5


@pytest.mark.parametrize("rows,C,T", [((18944, 18944), 3584, 24), ((18944, 18944), 3584, 32), ((18945, 3, 18950), 3584, 31), ((60001,), 2112, 32), ((7003,) * 8, 3008, 27), ((4000, 50003, 2), 3584, 17)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_sums_that_do_not_fit_at_once(rows, C, T):
    """Decode batches: rows a part at a time in the workspace there is are the bits of the whole product, also through the entry point that has 16 MB behind
    its header, and nothing behind the workspace is touched."""
    lins = [to_device(synth(R, C, 8, 16, 1, 1, seed=R + T), stream=False) for R in rows]
    mats, R = _mats(lins), sum(rows)
    L, room = _lib.lib(), 16 << 20
    assert L.sq_workspace_bytes(mats, len(lins), T, 2) > room
    x = rand_x(T, C, torch.bfloat16, seed=T)
    x[2, 5] = float("inf")
    x = x.cuda()
    want, y = (torch.full((T, R), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    _call(lins, x, want)
    linear_small(lins, x, y)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    args = (mats, len(lins), x.data_ptr(), _lib.SQ_BF16, C, y.data_ptr(), _lib.SQ_BF16, R, T)
    y.fill_(float("nan"))
    _lib.check(L.sq_linear_small_noalloc(*args, _lib.stream_ptr(x.device)))
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    ws = torch.full((room + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    y.fill_(float("nan"))
    _lib.check(L.sq_linear_small(*args, ws.data_ptr(), room, _lib.stream_ptr(x.device)))
    assert torch.equal(y.view(torch.int16), want.view(torch.int16)) and bool((ws[room:] == 0x5A).all())


@pytest.mark.parametrize("R,C,d,bits,G,M,T", [(99, 64, 8, 16, 1, 1, 16), (99, 64, 8, 16, 1, 1, 129), (99, 72, 8, 16, 1, 1, 20), (99, 64, 8, 16, 2, 1, 20), (99, 64, 8, 16, 1, 2, 20),
                                              (99, 64, 8, 15, 1, 1, 20), (99, 64, 4, 16, 1, 1, 20)])
def test_what_it_refuses(R, C, d, bits, G, M, T):
    f = _lib.lib().sq_plane_product_for_tests
    f.restype = _i64
    lin = to_device(synth(R, C, d, bits, G, M, seed=2), stream=False)
    assert f(_mats([lin]), 1, _p(None), 1, _i64(C), _p(None), 1, _i64(R), T, _p(None), _p(None)) < 0
