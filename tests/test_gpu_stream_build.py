"""The load-time layouts built on the GPU are the host builder's, byte for byte, and so is the relabelling."""

import ctypes
import math

import numpy as np
import pytest
import torch

from quantexperiments_amd import _lib
from quantexperiments_amd.kernels import build_stream, linear_small, prepare_stack
from quantexperiments_amd.packed import pack_bits
from tests.helpers import rand_x, rel_max_err, synth, to_device

pytestmark = pytest.mark.gpu

# R, C, d, bits, G, M, runs, tags
CASES = [(1, 64, 8, 16, 1, 1, 0, "any"), (65, 3584, 8, 16, 1, 1, 2, "any"), (200, 3976, 8, 13, 1, 1, 0, "any"), (64, 3968, 8, 14, 1, 1, 1, "any"),
         (300, 5120, 8, 16, 1, 16, 3, "any"), (130, 8 * 4100, 8, 16, 1, 1, 1, "any"), (70, 8 * 4064, 8, 13, 1, 1, 1, "one"), (90, 1024, 8, 12, 4, 1, 2, "any"),
         (40, 512, 8, 15, 2, 3, 0, "low"), (129, 17408, 8, 16, 1, 1, 0, "low"), (17, 640, 4, 10, 1, 1, 0, "any"), (16, 384, 4, 12, 1, 1, 0, "any"),
         (31, 896, 4, 8, 2, 1, 0, "any"),
         # the longest run there is, runs of one and of several column orders with a short last group, two runs of one order
         (6144, 256, 8, 13, 1, 1, 1, "any"), (6000, 264, 8, 14, 1, 3, 1, "low"), (1030, 64, 8, 16, 1, 16, 2, "one"), (6145, 128, 8, 13, 1, 1, 1, "low"),
         # entries of a lane below, at and beyond what a wave's registers hold; a second part that begins at an odd chunk
         (40, 8 * 63, 8, 16, 1, 1, 1, "one"), (33, 8 * 64, 8, 14, 1, 1, 1, "one"), (70, 8 * 65, 8, 15, 1, 1, 1, "one"),
         (66, 8 * 4069, 8, 16, 1, 1, 1, "any"), (21, 8 * 4069, 8, 14, 1, 1, 1, "low")]


@pytest.mark.parametrize("R,C,d,bits,G,M,runs,how", CASES)
def test_device_builder_writes_the_host_builders_bytes(R, C, d, bits, G, M, runs, how):
    g = torch.Generator().manual_seed(R * 7 + C)
    n = C // d
    top = {"any": 1 << bits, "low": 1 << (bits - 2), "one": 1}[how]
    words = pack_bits(torch.randint(0, top, (R, n), generator=g), bits)
    mask = torch.randint(0, M, (R,), generator=g).to(torch.uint8) if M > 1 else None
    book = (torch.randint(0, G, (R,), generator=g).to(torch.uint8), G) if G > 1 else None
    want, r0, g0 = build_stream(words, C, d, bits, mask, runs, row_book=book)
    got, r1, g1 = build_stream(words.cuda(), C, d, bits, mask, runs, row_book=None if book is None else (book[0].cuda(), G))
    assert (r0, g0) == (r1, g1) and want is not None
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("R,C,bits,G", [(3, 64, 16, 1), (70, 1000, 13, 1), (65, 3584, 16, 1), (90, 1032, 14, 4), (33, 264, 12, 2)])
def test_device_relabelling(R, C, bits, G):
    L = _lib.lib()
    g = torch.Generator().manual_seed(bits)
    n = C // 8
    tags = (torch.rand(R, n, generator=g) ** 3 * (1 << bits)).long().clamp_(max=(1 << bits) - 1)
    words = pack_bits(tags, bits)
    book = torch.randint(0, G, (R,), generator=g).to(torch.uint8)
    bp = book.data_ptr() if G > 1 else None
    want = np.zeros(G << bits, np.uint16)
    _lib.check(L.sq_codebook_balance_books(words.data_ptr(), R, words.shape[1], C, 8, bits, G, bp, want.ctypes.data))
    wd, bd = words.cuda(), book.cuda()
    counts = torch.empty(G << bits, dtype=torch.int32, device="cuda")
    remap = np.zeros(G << bits, np.uint16)
    args = (wd.data_ptr(), R, words.shape[1], C, 8, bits, G, bd.data_ptr() if G > 1 else None)
    _lib.check(L.sq_codebook_balance_device(*args, counts.data_ptr(), remap.ctypes.data, _lib.stream_ptr(wd.device)))
    assert np.array_equal(remap, want)
    rd = torch.from_numpy(remap.view(np.int16)).cuda()
    _lib.check(L.sq_codebook_relabel_device(*args, rd.data_ptr(), _lib.stream_ptr(wd.device)))
    at = tags.numpy() + (book.numpy().astype(np.int64) << bits)[:, None] if G > 1 else tags.numpy()
    assert torch.equal(wd.cpu(), pack_bits(torch.from_numpy(want[at].astype(np.int64)), bits))
    m = ctypes.c_void_p()
    assert L.sq_stream_plan_device(None, R, 1, C, 8, bits, G, None, None, 0, None, ctypes.byref(m), ctypes.byref(ctypes.c_size_t()),
                                   ctypes.byref(ctypes.c_size_t()), ctypes.byref(ctypes.c_int32()), ctypes.byref(ctypes.c_int32()), None) == _lib.SQ_EINVAL


def _counted(R, n, bits, how, g):
    """Tags [R, n] whose codewords are used: evenly; by a power law (counts of two and three bytes); only the first few (the rest
    not at all); each a different number of times (more of those than one list of runs holds)."""
    K = 1 << bits
    if how == "any":
        return torch.randint(0, K, (R, n), generator=g)
    if how == "zipf":
        return (torch.rand(R, n, generator=g, dtype=torch.float64).mul_(-math.log(K)).exp_() * K).long().clamp_(max=K - 1)
    if how == "few":
        return torch.randint(0, 5, (R, n), generator=g) * 3
    t = torch.repeat_interleave(torch.arange(6300), torch.arange(6300))
    t = torch.cat([t, torch.full((R * n - t.numel(),), K - 1)])
    return t[torch.randperm(t.numel(), generator=g)].view(R, n)


@pytest.mark.parametrize("R,C,bits,G,W,how", [(1, 8, 13, 1, 1, "any"), (70, 1000, 13, 1, 53, "zipf"), (65, 3584, 16, 1, 224, "any"), (600, 3584, 16, 1, 224, "zipf"),
                                              (90, 1032, 14, 4, 57, "zipf"), (33, 264, 12, 2, 13, "any"), (300, 512, 15, 2, 30, "few"),
                                              (4900, 32400, 16, 1, 2025, "each")])
def test_device_rebalance(R, C, bits, G, W, how):
    L, g, n = _lib.lib(), torch.Generator().manual_seed(bits + R), C // 8
    tags = _counted(R, n, bits, how, g)
    words = torch.full((R, W), -1, dtype=torch.int32)
    need = (n * bits + 31) // 32
    words[:, :need] = pack_bits(tags, bits)                     # (W > need: words behind the tags, which stay)
    book = torch.randint(0, G, (R,), generator=g).to(torch.uint8)
    table = torch.randn(G << bits, 8, generator=g).half()
    remap = np.zeros(G << bits, np.uint16)
    _lib.check(L.sq_codebook_balance_books(words.data_ptr(), R, W, C, 8, bits, G, book.data_ptr() if G > 1 else None, remap.ctypes.data))
    new = torch.from_numpy(remap.astype(np.int64))
    at = tags + (book.long() << bits)[:, None] if G > 1 else tags
    want = words.clone()
    want[:, :need] = pack_bits(new[at], bits)
    moved = torch.empty_like(table)
    moved[(torch.arange(G << bits) >> bits << bits) + new] = table
    dev = [t.cuda() for t in (words, table, book)]
    m = _lib.SqMatrix(dev[0].data_ptr(), dev[1].data_ptr(), None, dev[2].data_ptr() if G > 1 else None, None, None, None, R, C, 8, bits, G, 1, W, 0, None, 0, 0)
    mats = _lib.matrix_array([m] * 9)                           # (more than a launch takes)
    out = [(torch.empty_like(dev[0]), torch.empty_like(dev[1])) for _ in range(9)]
    ptrs = [(ctypes.c_void_p * 9)(*(o[k].data_ptr() for o in out)) for k in (0, 1)]
    scratch = torch.empty(L.sq_codebook_rebalance_bytes(mats, 9), dtype=torch.uint8, device="cuda")
    args = (mats, 9, *ptrs, scratch.data_ptr())
    assert L.sq_codebook_rebalance_device(*args, scratch.numel() - 1, None) == _lib.SQ_EWORKSPACE
    _lib.check(L.sq_codebook_rebalance_device(*args, scratch.numel(), _lib.stream_ptr(dev[0].device)))
    for w, t in out:
        assert torch.equal(w.cpu(), want) and torch.equal(t.cpu(), moved)


@pytest.mark.parametrize("G", [2, 4])
def test_unknown_codebooks_are_refused_before_a_launch(G):
    L, R, C, bits = _lib.lib(), 40, 512, 14
    words = torch.zeros(R, C // 8 * bits // 32, dtype=torch.int32, device="cuda")
    book = torch.zeros(R, dtype=torch.uint8, device="cuda")
    book[R - 1] = G
    counts = torch.full((G << bits,), -1, dtype=torch.int32, device="cuda")
    remap = np.zeros(G << bits, np.uint16)
    args = (words.data_ptr(), R, words.shape[1], C, 8, bits, G, book.data_ptr())
    assert L.sq_codebook_balance_device(*args, counts.data_ptr(), remap.ctypes.data, _lib.stream_ptr(words.device)) == _lib.SQ_EINVAL
    assert b"row 39 names codebook" in L.sq_last_error()
    plan, n, k, r, g = ctypes.c_void_p(), ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_int32(), ctypes.c_int32()
    assert L.sq_stream_counts_bytes(R, C, 8, bits, G) <= counts.numel() * 4
    assert L.sq_stream_plan_device(*args, None, 0, counts.data_ptr(), ctypes.byref(plan), ctypes.byref(n), ctypes.byref(k), ctypes.byref(r),
                                   ctypes.byref(g), _lib.stream_ptr(words.device)) == _lib.SQ_EINVAL and not plan.value
    assert bool((counts == -1).all())
    with pytest.raises(ValueError, match="row_book"):
        build_stream(words, C, 8, bits, row_book=(book, G))


@pytest.mark.parametrize("rows,C,d,bits,G,M", [((300,), 1024, 8, 16, 1, 1), ((600, 65, 66), 3584, 8, 16, 1, 1), ((130, 40), 512, 8, 14, 2, 3),
                                               ((40,), 8 * 4069, 8, 13, 1, 1), ((300,), 3584, 4, 12, 1, 1), ((300,), 896, 4, 8, 2, 1)])
def test_layouts_are_whole_when_they_are_handed_back(rows, C, d, bits, G, M):
    """Built under one stream, multiplied on another that waits for nothing where the layout is a slice stream."""
    ss = [synth(R, C, d, bits, G, M, seed=R) for R in rows]
    lins = [to_device(s, stream=False) for s in ss]             # (the tensors themselves, in place before the side stream begins)
    x = rand_x(1, C, torch.float16, seed=1).cuda()
    y = torch.zeros(1, sum(rows), device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side := torch.cuda.Stream()):
        if len(lins) == 1:
            lins[0].wants_stream = d == 8
            lins[0].build_stream()
            lins[0].stream_tiled = d == 4
        else:
            for lin in lins:
                lin.wants_stream = True
            prepare_stack(lins)
        assert side.query() or d == 4
    assert all(lin.stream is not None for lin in lins)
    if d == 4:                                                  # (a tile-major copy is ordered by its stream)
        torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        linear_small(lins, x, y)
    torch.cuda.synchronize()
    want = np.concatenate([x.cpu().double().numpy() @ s.decode().astype(np.float64).T for s in ss], axis=1)
    assert rel_max_err(y.cpu().numpy(), want) < 1e-5            # (exact products, fp32 sums)


def test_a_relabelling_that_failed_is_done_again(monkeypatch):
    """The launch fails once: nothing of the matrices has changed, and the next build relabels them."""
    L, ss = _lib.lib(), [synth(R, 1024, 8, 16, seed=R) for R in (200, 70)]
    want, lins = [[to_device(s, stream="later") for s in ss] for _ in range(2)]
    prepare_stack(want)
    before = [(m.words, m.table) for m in lins]
    with monkeypatch.context() as mp:
        mp.setattr(L, "sq_codebook_rebalance_device", lambda *a: _lib.SQ_ELAUNCH)
        with pytest.raises(RuntimeError):
            prepare_stack(lins)
    assert all(m.stream is None and not m.relabelled and m.words is w and m.table is t for m, (w, t) in zip(lins, before))
    prepare_stack(lins)
    for m, w, (words, _) in zip(lins, want, before):
        assert not torch.equal(m.words, words) and m.relabelled and torch.equal(m.words, w.words)
        assert torch.equal(m.table, w.table) and torch.equal(m.stream, w.stream) and m.stream_runs == w.stream_runs


@pytest.mark.parametrize("bits", [13, 16])
@pytest.mark.parametrize("most", [1, 2, 3, 7, 8, 15, 16, 31, 32, 63, 64, 127, 128, 255, 256, 300])
def test_dealing_by_largest_count(most, bits):
    """Every width of the digit that the codewords are sorted by, and two digits; codewords without tags are one long step."""
    L, g, R, C = _lib.lib(), torch.Generator().manual_seed(most), 40, 8 * 200
    pool = torch.randperm(1 << bits, generator=g)[:R * 200 // most + 1].repeat_interleave(torch.randint(1, most + 1, (R * 200 // most + 1,), generator=g))
    tags = torch.cat([torch.full((most,), int(pool[0])), pool[pool != pool[0]], torch.arange(R * 200) % (1 << bits)])[:R * 200]
    assert most == 1 or int(torch.bincount(tags).max()) >= most
    tags = tags[torch.randperm(R * 200, generator=g)].view(R, 200)
    words = pack_bits(tags, bits)
    remap = np.zeros(1 << bits, np.uint16)
    _lib.check(L.sq_codebook_balance_books(words.data_ptr(), R, words.shape[1], C, 8, bits, 1, None, remap.ctypes.data))
    wd, td = words.cuda(), torch.randn(1 << bits, 8, generator=g).half().cuda()
    mats = _lib.matrix_array([_lib.SqMatrix(wd.data_ptr(), td.data_ptr(), None, None, None, None, None, R, C, 8, bits, 1, 1, words.shape[1], 0, None, 0, 0)])
    wo, to = torch.empty_like(wd), torch.empty_like(td)
    scratch = torch.empty(L.sq_codebook_rebalance_bytes(mats, 1), dtype=torch.uint8, device="cuda")
    _lib.check(L.sq_codebook_rebalance_device(mats, 1, *((ctypes.c_void_p * 1)(t.data_ptr()) for t in (wo, to)), scratch.data_ptr(), scratch.numel(), None))
    new = torch.from_numpy(remap.astype(np.int64))
    assert torch.equal(wo.cpu(), pack_bits(new[tags], bits))
    assert torch.equal(to.cpu()[new], td.cpu())
