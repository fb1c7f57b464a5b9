"""16-bit tags of width 8 decoded a column of the codebook at a time for the tile GEMM: weights and activations in plane order bit by bit,
rows that end within a workgroup's step, one row, pieces of very different sizes, activations with a row stride, and whole products."""

import ctypes

import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import linear_gemm
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu


_i64 = ctypes.c_int64


def _p(t):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _plane_order(a):
    """[rows, chunks * 8] -> [rows, 8 * chunks]"""
    return a.view(a.shape[0], -1, 8).transpose(1, 2).reshape(a.shape[0], -1)


@pytest.mark.parametrize("rows,C,T,dtype", [
    ((1,), 64, 1, torch.bfloat16), ((1, 1, 1, 1, 1, 1, 1, 1), 64, 3, torch.float16), ((63, 65), 64, 33, torch.bfloat16), ((4097, 1, 130), 192, 65, torch.float16),
    ((16384,), 512, 100, torch.bfloat16), ((16385, 3), 576, 31, torch.float16), ((40001,), 320, 7, torch.bfloat16), ((257, 1023, 5000), 3584, 64, torch.bfloat16)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_decode_is_the_codewords_in_plane_order(rows, C, T, dtype):
    ss = [synth(R, C, 8, 16, 1, 1, seed=R + i) for i, R in enumerate(rows)]
    lins = [to_device(s, stream=False) for s in ss]
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()
    guard = 64
    out = torch.full((sum(rows) * C + guard,), 7.0, dtype=torch.float16, device="cuda")
    xout = torch.full((T * C + guard,), 7.0, dtype=torch.float16, device="cuda")
    planes = torch.empty(len(rows) << 19, dtype=torch.float16, device="cuda")
    rc = _lib.lib().sq_planes_for_tests(_lib.matrix_array([m.descriptor() for m in lins]), len(lins), _p(out), _p(planes), _p(xd), _lib.DTYPES[dtype], _i64(C + 8), T,
                                        _p(xout), _p(None))
    torch.cuda.synchronize()
    assert rc == 0
    ref = torch.cat([torch.from_numpy(s.table)[torch.from_numpy(s.tags)].reshape(s.R, C) for s in ss])
    assert torch.equal(out[:-guard].view(-1, C).cpu().view(torch.int16), _plane_order(ref).view(torch.int16))
    assert torch.equal(xout[:-guard].view(T, C).cpu().view(torch.int16), _plane_order(x[:, :C].half()).view(torch.int16))
    assert bool((out[-guard:] == 7).all()) and bool((xout[-guard:] == 7).all())


PRODUCTS = [((3001, 3000), 3584, 900, (7, 7)), ((26003,), 1280, 520, (7, 7)), ((1000, 250, 249), 4032, 700, (7, 7)), ((18944,), 1600, 1030, (7, 6)), ((1100,), 1024, 2000, (6, 6))]


# kernels: the one that bf16 and that fp16 activations take, 7 where the codebooks go in columns, 6 a codeword at a time (too little to gain)
@pytest.mark.parametrize("rows,C,T,kernels", PRODUCTS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_products(rows, C, T, kernels, dtype):
    ss = [synth(R, C, 8, 16, 1, 1, seed=R) for R in rows]
    lins = [to_device(s, stream=False) for s in ss]
    mats = _lib.matrix_array([m.descriptor(sum(rows[:i])) for i, m in enumerate(lins)])
    kernel = _lib.lib().sq_gemm_kernel_for_tests(mats, len(lins), T, _lib.DTYPES[dtype], (ctypes.c_float * 3)())
    assert torch.cuda.get_device_properties(0).multi_processor_count != 256 or kernel == kernels[dtype == torch.float16]
    x = torch.zeros(T, C + 8, dtype=dtype)
    x[:, :C] = rand_x(T, C, dtype, seed=T)
    xd = x.cuda()[:, :C]
    y = torch.zeros(T, sum(rows) + 1, dtype=torch.float32, device="cuda")
    linear_gemm(lins, xd, y[:, :sum(rows)])
    ref = torch.cat([xd.double() @ torch.from_numpy(s.decode()).cuda().double().T for s in ss], dim=1)
    # products of fp16 values are exact in fp32, whose sums of C terms round at 2^-24 of a partial sum: below sqrt(C) 2^-24 of the largest result
    assert rel_max_err(y[:, :sum(rows)].cpu().numpy(), ref.cpu().numpy()) < 1e-5 and not y[:, sum(rows):].any()


@pytest.mark.parametrize("change", ["width", "orders", "books", "bits", "ragged"])
def test_other_formats_are_refused(change):
    R, C, d, bits, G, M = {"width": (9, 64, 4, 16, 1, 1), "orders": (9, 64, 8, 16, 1, 4), "books": (9, 64, 8, 16, 2, 1), "bits": (9, 64, 8, 15, 1, 1),
                           "ragged": (9, 72, 8, 16, 1, 1)}[change]
    lins = [to_device(synth(9, C, 8, 16, 1, 1, seed=1), stream=False), to_device(synth(R, C, d, bits, G, M, seed=2), stream=False)]
    null = _p(None)
    rc = _lib.lib().sq_planes_for_tests(_lib.matrix_array([m.descriptor() for m in lins]), 2, null, null, null, 1, _i64(C), 0, null, null)
    assert rc != 0
