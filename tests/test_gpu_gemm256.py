"""The 256 x 256 tile GEMM where its loop and its tile walk have edges: one to four slabs of K, partial tiles both ways, more
than one super-column of token tiles, unaligned outputs, and stacks with more pieces than one launch scales."""

import numpy as np
import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import gemm_dense, linear_gemm
from quantexperiments_amd.vllm_ext import core
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,R,C", [(33, 1, 64), (256, 256, 128), (257, 300, 192), (64, 511, 256), (2305, 260, 64), (4200, 70, 128)])
@pytest.mark.parametrize("dtype,pad", [(torch.bfloat16, 0), (torch.float16, 8), (torch.float16, 3), (torch.float32, 0)])
def test_tile_edges(T, R, C, dtype, pad):
    g = torch.Generator().manual_seed(T + R)
    x, w = torch.randn(T, C, generator=g).half(), torch.randn(R, C, generator=g).half()
    ref = (x.float() @ w.float().T).numpy().astype(np.float64)
    y = torch.full((T, (R + 7) // 8 * 8 + pad), float("nan"), dtype=dtype, device="cuda")
    gemm_dense(w.cuda(), x.cuda(), y[:, :R])
    assert rel_max_err(y[:, :R].float().cpu().numpy(), ref) < {torch.float32: 1e-5, torch.float16: 1e-3, torch.bfloat16: 5e-3}[dtype]
    assert torch.isnan(y[:, R:]).all()


@pytest.mark.parametrize("n", [4, 5])
def test_stack_of_pieces(n):
    ss = [synth(40 + 3 * i, 128, 8, 13, seed=i) for i in range(n)]
    x = rand_x(300, 128, torch.bfloat16, seed=n)
    y = torch.empty(300, sum(s.R for s in ss), dtype=torch.float32, device="cuda")
    linear_gemm([to_device(s, stream=False) for s in ss], x.cuda(), y)
    ref = np.concatenate([x.float().numpy().astype(np.float64) @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.cpu().numpy(), ref) < 1e-3


@pytest.mark.parametrize("n", [5, 8, 9, 17])
@pytest.mark.parametrize("d,bits,M", [(8, 16, 1), (8, 16, 3), (4, 12, 1)])
def test_long_stacks(n, d, bits, M):
    """Stacks of more pieces than a launch scales: a product per eight, each piece with its own scales and at its own columns; and
    their workspace, a joint product's per eight pieces."""
    L, T, C = _lib.lib(), 400, 512
    ss = [synth(33 + 8 * i, C, d, bits, 1, M, seed=i) for i in range(n)]
    lins = [to_device(s, stream=False) for s in ss]
    x = rand_x(T, C, torch.bfloat16, seed=n)
    rows = sum(s.R for s in ss)
    y = torch.full((T, rows), float("nan"), dtype=torch.float32, device="cuda")
    linear_gemm(lins, x.cuda(), y)
    ref = np.concatenate([x.float().numpy().astype(np.float64) @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.cpu().numpy(), ref) < 1e-3
    dense = lambda of: sum((s.R * C * 2 + 255) // 256 * 256 for s in of)
    off, mats = 0, []
    for lin in lins:
        mats.append(lin.descriptor(off))
        off += lin.R
    need = L.sq_workspace_bytes(_lib.matrix_array(mats), n, T, 1) - _lib.WS_HEADER - T * C * 2
    most = max(dense(ss[i:i + 8]) for i in range(0, n, 8))
    assert need >= most and need - most < 64 << 20


@pytest.mark.parametrize("T,R,C", [
    (129, 300, 64), (65, 257, 320), (333, 2000, 2048), (200, 890, 8960),      # tiles of 128 token rows, also split along K
    (190, 60000, 64), (185, 60001, 320), (300, 34000, 4096),        # of 192: one slab, five, two rounds with a split last one
    (250, 65700, 192), (257, 33000, 64), (510, 34000, 4096)])       # of 256
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_tile_heights(T, R, C, dtype):
    g = torch.Generator(device="cuda").manual_seed(T + R)
    x, w = (torch.randn(n, C, generator=g, device="cuda").half() for n in (T, R))
    y = torch.full((T, R + 8), float("nan"), dtype=dtype, device="cuda")
    gemm_dense(w, x, y[:, :R])
    ref = x.double() @ w.double().T
    # C roundings to fp32, in any order, each at most 2^-24 of a partial sum; those of C products of unit normals stay below
    # 5 sqrt(C), and roundings of random sign add up to less than 6 sqrt(C / 3) of them: 17.4 C 2^-24. A slab
    # left out is off by 8.
    bound = 17.4 * C * 2.0 ** -24 + (2.0 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0.0)
    assert ((y[:, :R].double() - ref).abs() <= bound).all()
    assert torch.isnan(y[:, R:]).all()


@pytest.mark.parametrize("T,R,C", [
    (512, 70400, 64), (520, 70000, 72), (512, 40960, 192), (700, 33000, 328),        # tiles of 256 token rows: one to six slabs, whole and broken
    (192, 140000, 64), (380, 70000, 136), (128, 140032, 64), (121, 140000, 200)])    # of 192 and 128
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tiles_one_after_another(T, R, C, dtype):
    """Several tiles to a workgroup, whole ones and ones at the matrix' edges in turn, whose 16-bit results leave in 16-byte pieces
    while the next tile's slabs arrive."""
    g = torch.Generator(device="cuda").manual_seed(T + R)
    x, w = (torch.randn(n, C, generator=g, device="cuda").half() for n in (T, R))
    y = torch.full((T, R + 8), float("nan"), dtype=dtype, device="cuda")
    for _ in range(3):
        gemm_dense(w, x, y[:, :R])
    ref = x.double() @ w.double().T
    bound = 17.4 * C * 2.0 ** -24 + 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * ref.abs()     # as in test_tile_heights
    assert ((y[:, :R].double() - ref).abs() <= bound).all()
    assert torch.isnan(y[:, R:]).all()


@pytest.mark.parametrize("limit", [0, 150 * 512 * 2, 1 << 30])
@pytest.mark.parametrize("T", [40, 800])
def test_dequant_route_in_groups_of_pieces(limit, T, monkeypatch):
    monkeypatch.setattr(core, "JOINT_BYTES", limit)
    monkeypatch.setattr(core, "JOINT_BYTES_MANY_ROWS", limit)
    ss = [synth(R, 512, 8, 16, 1, 3, seed=R) for R in (100, 40, 10, 141, 9)]
    ps = core.PackedShards([to_device(s, stream=False) for s in ss], large="dequant")
    x = rand_x(T, 512, torch.bfloat16, seed=T)
    y = ps.forward(x.cuda())
    ref = np.concatenate([x.float().numpy().astype(np.float64) @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.float().cpu().numpy(), ref) < 5e-3


@pytest.mark.parametrize("T,R,C", [
    (33, 70, 8), (64, 300, 56), (129, 257, 72), (200, 890, 8968), (333, 2000, 2040),      # tiles of 128 token rows, also split along K
    (190, 60000, 88), (300, 34000, 4120), (250, 65700, 200), (510, 34000, 4104)])       # of 192 and 256
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_broken_slabs(T, R, C, dtype):
    """Rows whose last slab of 64 columns is not whole, between columns that hold NaN."""
    g = torch.Generator(device="cuda").manual_seed(T + R)
    x, w = (torch.full((n, C + 72), float("nan"), dtype=torch.float16, device="cuda") for n in (T, R))
    for t in (x, w):
        t[:, :C] = torch.randn(t.shape[0], C, generator=g, device="cuda").half()
    y = torch.full((T, R + 8), float("nan"), dtype=dtype, device="cuda")
    gemm_dense(w[:, :C], x[:, :C], y[:, :R])
    ref = x[:, :C].double() @ w[:, :C].double().T
    bound = 17.4 * C * 2.0 ** -24 + (2.0 ** -8 * ref.abs() if dtype == torch.bfloat16 else 0.0)     # as in test_tile_heights
    assert ((y[:, :R].double() - ref).abs() <= bound).all()
    assert torch.isnan(y[:, R:]).all()


@pytest.mark.parametrize("large", ["fused", "dequant"])
@pytest.mark.parametrize("d,bits,G,M,C,T", [(4, 10, 4, 1, 1360, 300), (4, 12, 1, 1, 2056, 700), (8, 16, 1, 1, 1032, 260), (8, 16, 1, 3, 1096, 600), (4, 8, 1, 1, 1992, 257)])
def test_broken_rows_in_tiles(d, bits, G, M, C, T, large):
    ss = [synth(R, C, d, bits, G, M, seed=R) for R in (100, 41, 300)]
    ps = core.PackedShards([to_device(s, stream=False) for s in ss], large=large)
    x = rand_x(T, C, torch.bfloat16, seed=T)
    y = ps.forward(x.cuda())
    ref = np.concatenate([x.float().numpy().astype(np.float64) @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.float().cpu().numpy(), ref) < 5e-3


@pytest.mark.parametrize("T,R,C", [(130, 2, 64), (257, 299, 192), (700, 1026, 128), (300, 700, 4160), (2049, 9001, 64), (1500, 16514, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_of_results_without_16_byte_stores(T, R, C, dtype):
    """16-bit results whose rows allow stores of 4 bytes or 2: the same products and the same rounding as rows that allow 16, so the same
    bits; one tile per workgroup, several, parts of tiles; nothing is written beside the rows."""
    g = torch.Generator(device="cuda").manual_seed(T + R)
    x = torch.randn(T, C, device="cuda", generator=g).half()
    w = torch.randn(R, C, device="cuda", generator=g).half()
    want = torch.zeros(T, (R + 15) // 8 * 8, dtype=dtype, device="cuda")
    gemm_dense(w, x, want[:, :R])
    for ld, off in ((R + 3 + (R + 3) % 2, 2), (R + 4 + (R + 5) % 2, 0), (R + 4, 1)):
        y = torch.full((T * ld + 16,), 5.0, dtype=dtype, device="cuda")
        rows = y[off:off + T * ld].view(T, ld)
        gemm_dense(w, x, rows[:, :R])
        assert torch.equal(rows[:, :R], want[:, :R]), (ld, off)
        assert bool((rows[:, R:] == 5.0).all()) and bool((y[:off] == 5.0).all()) and bool((y[off + T * ld:] == 5.0).all())
