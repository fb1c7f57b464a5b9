"""The C-ABI library loads, exports every function include/sqhip.h declares, and rejects bad
arguments on the host before any GPU work.  CPU only: no kernel is launched here."""

import ctypes
import re
from pathlib import Path

import pytest

from quantexperiments_amd import _lib

ROOT = Path(__file__).resolve().parents[1]


def _declared():
    text = (ROOT / "include" / "sqhip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sq_[a-z0-9_]+)\s*\(", text)))


def test_header_and_loader_agree():
    assert _declared() == sorted(_lib.EXPORTS)


def test_library_exports_every_declared_symbol():
    L = _lib.lib()
    for name in _declared():
        assert getattr(L, name) is not None, name
    assert L.sq_version() == 109


def test_struct_layout_matches_header():
    # 7 pointers + 8 int32 + 1 pointer + 2 int32
    assert ctypes.sizeof(_lib.SqMatrix) == 7 * 8 + 8 * 4 + 8 + 8
    assert _lib.SqMatrix.R.offset == 56 and _lib.SqMatrix.y_off.offset == 56 + 28 and _lib.SqMatrix.stream.offset == 88 and _lib.SqMatrix.stream_groups.offset == 100
    # sq_producer: int32 mode, float eps, 6 pointers, 2 int64
    assert ctypes.sizeof(_lib.SqProducer) == 8 + 6 * 8 + 2 * 8
    assert _lib.SqProducer.eps.offset == 4 and _lib.SqProducer.h_in.offset == 8 and _lib.SqProducer.x_out.offset == 48 and _lib.SqProducer.ld_in.offset == 64


def test_host_side_argument_checks():
    L = _lib.lib()
    m = _lib.SqMatrix()                       # all null
    assert L.sq_dequant(ctypes.byref(m), None, _lib.SQ_F32, 0, 0, 0, None) == _lib.SQ_EINVAL
    assert b"null" in L.sq_last_error()
    m = _lib.SqMatrix(0x1000, 0x2000, 0x3000, None, None, None, None, 4, 30, 4, 8, 1, 1, 2, 0)
    assert L.sq_dequant(ctypes.byref(m), None, _lib.SQ_F32, 30, 0, 4, None) == _lib.SQ_EINVAL   # C % d
    m.C = 32
    m.bits = 17
    assert L.sq_dequant(ctypes.byref(m), None, _lib.SQ_F32, 32, 0, 4, None) == _lib.SQ_EINVAL
    m.bits = 8
    m.W = 1                                   # 8 tags of 8 bits need 2 words
    assert L.sq_dequant(ctypes.byref(m), None, _lib.SQ_F32, 32, 0, 4, None) == _lib.SQ_EINVAL
    m.W = 2
    assert L.sq_dequant(ctypes.byref(m), None, _lib.SQ_F32, 32, 3, 9, None) == _lib.SQ_EINVAL   # rows outside
    assert L.sq_dequant(ctypes.byref(m), None, _lib.SQ_F32, 32, 2, 2, None) == _lib.SQ_OK       # empty range
    m.M = 4                                   # masks without row_mask / perms
    arr = _lib.matrix_array([m])
    assert L.sq_linear_small(arr, 1, 0x4000, _lib.SQ_BF16, 32, 0x5000, _lib.SQ_BF16, 4, 1, None, 0, None) == _lib.SQ_EINVAL
    m.M = 1
    arr = _lib.matrix_array([m])
    assert L.sq_linear_small(arr, 1, 0x4000, _lib.SQ_F32, 32, 0x5000, _lib.SQ_F32, 4, 1, None, 0, None) == _lib.SQ_EINVAL
    assert L.sq_linear_small(arr, 1, 0x4000, _lib.SQ_BF16, 32, 0x5000, _lib.SQ_BF16, 4, 33, None, 0, None) == _lib.SQ_EINVAL
    assert L.sq_linear_small(arr, 1, 0x4000, _lib.SQ_BF16, 32, 0x5000, _lib.SQ_BF16, 4, 0, None, 0, None) == _lib.SQ_OK
    assert L.sq_linear_gemm(arr, 1, 0x4000, _lib.SQ_BF16, 16, 0x5000, _lib.SQ_BF16, 4, 64, None, 0, None) == _lib.SQ_EINVAL
    assert L.sq_gemm_dense(0x1000, 5, 32, 8, 32, 0x4000, _lib.SQ_F16, 32, 0x5000, _lib.SQ_F16, 8, 4, None) == _lib.SQ_EINVAL
    with pytest.raises(_lib.SqError):
        _lib.check(_lib.SQ_EINVAL)


def test_workspace_sizes_are_host_arithmetic():
    L = _lib.lib()
    plain = _lib.SqMatrix(0x1000, 0x2000, 0x3000, None, None, None, None, 64, 512, 8, 16, 1, 1, 32, 0)
    masked = _lib.SqMatrix(0x1000, 0x2000, 0x3000, None, 0x6000, 0x7000, None, 64, 512, 8, 16, 1, 16, 32, 0)
    assert L.sq_workspace_bytes(_lib.matrix_array([plain]), 1, 1, 0) == 0
    # 33 .. 64 rows of a matrix the matrix-core decode kernel takes: passes of 32 rows, its workspace (none here)
    assert L.sq_workspace_bytes(_lib.matrix_array([plain]), 1, 64, 1) == 0
    lds = _lib.SqMatrix(0x1000, 0x2000, 0x3000, None, None, None, None, 64, 512, 4, 12, 1, 1, 48, 0)
    assert L.sq_workspace_bytes(_lib.matrix_array([lds]), 1, 224, 1) == 0          # codebook in LDS: up to 224 rows
    assert L.sq_workspace_bytes(_lib.matrix_array([lds]), 1, 225, 1) == _lib.WS_HEADER + 64 * 512 * 2 + 225 * 512 * 2
    # beyond: raw fp16 codewords of the largest piece + an fp16 copy of the activations
    assert L.sq_workspace_bytes(_lib.matrix_array([plain]), 1, 100, 1) == _lib.WS_HEADER + 64 * 512 * 2 + 100 * 512 * 2
    assert L.sq_workspace_bytes(_lib.matrix_array([plain]), 1, 2048, 1) == _lib.WS_HEADER + 64 * 512 * 2 + 2048 * 512 * 2
    assert L.sq_workspace_bytes(_lib.matrix_array([masked]), 1, 2, 0) == _lib.WS_HEADER + 16 * 2 * 512 * 2
    # which | 2: a workspace for these pieces alone has no header unless they keep partial sums there
    assert L.sq_workspace_bytes(_lib.matrix_array([masked]), 1, 2, 2) == 16 * 2 * 512 * 2
    assert L.sq_workspace_bytes(_lib.matrix_array([plain]), 1, 100, 3) == 64 * 512 * 2 + 100 * 512 * 2
    assert L.sq_workspace_bytes(_lib.matrix_array([masked]), 1, 100, 1) == _lib.WS_HEADER + 64 * 512 * 2 + 100 * 512 * 2
    # a matrix with a tag stream keeps its partial sums in the header and needs nothing behind it at decode time
    streamed = _lib.SqMatrix(0x1000, 0x2000, 0x3000, None, None, None, None, 64, 512, 8, 16, 1, 1, 32, 0, 0x8000, (1 << 16) | 1, 1)
    assert L.sq_workspace_bytes(_lib.matrix_array([streamed]), 1, 1, 0) == _lib.WS_HEADER
    assert L.sq_workspace_bytes(_lib.matrix_array([streamed]), 1, 8, 0) == _lib.WS_HEADER


def test_block32_entry_points_check_arguments_on_the_host():
    L = _lib.lib()
    bf, f32 = _lib.SQ_BF16, _lib.SQ_F32
    q, sc, x, y = 0x10000, 0x20000, 0x30000, 0x40000
    assert L.sq_q8_linear(q, sc, 64, 48, x, bf, 48, y, bf, 64, 1, None, 0, None) == _lib.SQ_EINVAL      # C % 32
    assert b"multiple of 32" in L.sq_last_error()
    assert L.sq_q8_linear(q + 4, sc, 64, 64, x, bf, 64, y, bf, 64, 1, None, 0, None) == _lib.SQ_EINVAL  # q alignment
    assert L.sq_q8_linear(None, sc, 64, 64, x, bf, 64, y, bf, 64, 1, None, 0, None) == _lib.SQ_EINVAL
    assert L.sq_q8_linear(q, sc, 64, 64, x, f32, 64, y, f32, 64, 1, None, 0, None) == _lib.SQ_EINVAL    # x dtype
    assert L.sq_q8_linear(q, sc, 64, 64, x, bf, 64, y, _lib.SQ_F16, 64, 1, None, 0, None) == _lib.SQ_EINVAL
    assert L.sq_q8_linear(q, sc, 64, 64, x, bf, 32, y, bf, 64, 2, None, 0, None) == _lib.SQ_EINVAL      # ldx < C
    assert L.sq_q8_linear(q, sc, 64, 64, x, bf, 64, y, bf, 63, 2, None, 0, None) == _lib.SQ_EINVAL      # ldy < V
    assert L.sq_q8_linear(q, sc, 64, 64, x, bf, 64, y, bf, 64, 0, None, 0, None) == _lib.SQ_OK          # no rows
    assert L.sq_q8_linear(q, sc, 0, 64, x, bf, 64, y, bf, 64, 4, None, 0, None) == _lib.SQ_OK           # no weights
    # more than 32 activation rows need the workspace sq_q8_workspace_bytes names
    assert L.sq_q8_linear(q, sc, 64, 64, x, bf, 64, y, bf, 64, 40, None, 0, None) == _lib.SQ_EWORKSPACE
    assert L.sq_q8_workspace_bytes(64, 64, 32) == 0
    assert L.sq_q8_workspace_bytes(64, 64, 40) == _lib.WS_HEADER + 64 * 64 * 2 + 40 * 64 * 2      # decoded rows + fp16 x
    assert L.sq_q8_workspace_bytes(64, 48, 40) == 0
    # 3 .. 320 rows with C % 256 == 0: an fp16 copy of the activations
    assert L.sq_q8_workspace_bytes(64, 256, 2) == 0
    assert L.sq_q8_workspace_bytes(64, 256, 3) == _lib.WS_HEADER + 3 * 256 * 2
    assert L.sq_q8_workspace_bytes(64, 1024, 4) == _lib.WS_HEADER + 4 * 1024 * 2
    assert L.sq_q8_workspace_bytes(64, 256, 8) == _lib.WS_HEADER + 8 * 256 * 2
    assert L.sq_q8_workspace_bytes(64, 256, 128) == _lib.WS_HEADER + 128 * 256 * 2
    assert L.sq_q8_workspace_bytes(64, 256, 320) == _lib.WS_HEADER + 320 * 256 * 2
    assert L.sq_q8_workspace_bytes(64, 256, 321) == _lib.WS_HEADER + 64 * 256 * 2 + 321 * 256 * 2
    assert L.sq_q8_linear(q, sc, 64, 256, x, bf, 256, y, bf, 64, 8, None, 0, None) == _lib.SQ_EWORKSPACE
    assert L.sq_q8_dequant(q, sc, 64, 64, y, f32, 64, 3, 65, None) == _lib.SQ_EINVAL                    # rows outside
    assert L.sq_q8_dequant(q, sc, 64, 64, y, f32, 32, 0, 4, None) == _lib.SQ_EINVAL                     # ld_out < C
    assert L.sq_q8_dequant(q, sc, 64, 64, y, 7, 64, 0, 4, None) == _lib.SQ_EINVAL
    assert L.sq_q8_dequant(q, sc, 64, 64, y, f32, 64, 5, 5, None) == _lib.SQ_OK
    assert L.sq_q4_embed(q, sc, 64, 64, x, -1, y, bf, 64, None) == _lib.SQ_EINVAL
    assert L.sq_q4_embed(q, sc, 64, 64, x + 4, 3, y, bf, 64, None) == _lib.SQ_EINVAL                    # ids alignment
    assert L.sq_q4_embed(q, sc, 64, 64, None, 3, y, bf, 64, None) == _lib.SQ_EINVAL
    assert L.sq_q4_embed(q, sc, 64, 64, x, 3, y, bf, 48, None) == _lib.SQ_EINVAL                        # ld_out < C
    assert L.sq_q4_embed(q, sc, 64, 64, x, 0, y, bf, 64, None) == _lib.SQ_OK


def test_neighbour_entry_points_check_arguments_on_the_host():
    L = _lib.lib()
    f16, bf, f32 = _lib.SQ_F16, _lib.SQ_BF16, _lib.SQ_F32
    p = 0x10000
    assert L.sq_addnorm(p, None, 64, None, 0, 0, p, f16, None, 1, 1, 0, 1e-6, p, f16, None) == _lib.SQ_EINVAL       # C = 0
    assert L.sq_addnorm(p, None, 64, None, 0, 0, p, f32, None, 1, 1, 64, 1e-6, p, f16, None) == _lib.SQ_EINVAL      # fp32 weights
    assert L.sq_addnorm(p, None, 64, p, f32, 64, p, f16, None, 1, 1, 64, 1e-6, p, f16, None) == _lib.SQ_EINVAL      # fp32 add
    assert L.sq_addnorm(None, None, 64, None, 0, 0, p, f16, None, 1, 1, 64, 1e-6, p, f16, None) == _lib.SQ_EINVAL   # no h_in
    assert L.sq_addnorm(p, None, 32, None, 0, 0, p, f16, None, 1, 2, 64, 1e-6, p, f16, None) == _lib.SQ_EINVAL      # ld_h < C
    assert L.sq_addnorm(p, p, 64, None, 0, 0, p, f16, p, 2, 1, 64, 1e-6, p, f16, None) == _lib.SQ_EINVAL            # in place with orders
    assert L.sq_addnorm(p, None, 64, None, 0, 0, p, f16, p, 0, 1, 64, 1e-6, p, f16, None) == _lib.SQ_EINVAL         # M = 0
    assert L.sq_addnorm(p, None, 64, None, 0, 0, p, f16, None, 1, 0, 64, 1e-6, None, f16, None) == _lib.SQ_OK       # no rows
    assert L.sq_silu_mul(p, p, f32, 64, None, 1, 1, 64, p, None) == _lib.SQ_EINVAL
    assert L.sq_silu_mul(p, None, bf, 64, None, 1, 1, 64, p, None) == _lib.SQ_EINVAL
    assert L.sq_silu_mul(p, p, bf, 64, None, 1, 0, 64, None, None) == _lib.SQ_OK
    pr = _lib.SqProducer()
    m = _lib.matrix_array([])
    assert L.sq_linear_small_from(m, 0, None, bf, p, bf, 64, 1, None, 0, None) == _lib.SQ_EINVAL                    # no producer
    pr.mode = 3
    assert L.sq_linear_small_from(m, 0, ctypes.byref(pr), bf, p, bf, 64, 1, None, 0, None) == _lib.SQ_EINVAL        # unknown mode
    pr.mode = _lib.SQ_FROM_SILU_MUL
    assert L.sq_linear_small_from(m, 0, ctypes.byref(pr), bf, p, bf, 64, 1, None, 0, None) == _lib.SQ_OK            # no pieces


def test_workspace_of_decoded_weights_is_bounded():
    """Ragged rows and column orders at 33 to 256 activation rows are decoded into the workspace, 192 MB of fp16 at a time."""
    L, step = _lib.lib(), 192 << 20

    def need(rows, C, d, bits, M, T, which=1):
        mats, off = [], 0
        for R in rows:
            mats.append(_lib.SqMatrix(0x10000, 0x20000, 0x30000, None, 0x50000 if M > 1 else None, 0x60000 if M > 1 else None, None, R, C, d, bits,
                                      1, M, (C // d * bits + 31) // 32, off))
            off += R
        return L.sq_workspace_bytes(_lib.matrix_array(mats), len(rows), T, which) - _lib.WS_HEADER

    for rows in ((18944, 18944), (40000,), (100, 90000, 7), (1000,) * 8, (300000,)):
        for d, bits in ((8, 16), (4, 12)):
            for T in (33, 128, 256):
                for C in (3592, 5128):
                    dense = sum(rows) * C * 2
                    assert min(dense, step // 2) <= need(rows, C, d, bits, 1, T) <= min(dense + 4096, step) + 8 * T * 128 * 256 * 4
    for rows in ((30000,), (20000, 10000), (1000,) * 8):
        for C in (5120, 5128):
            for T in (5, 16, 32):
                assert need(rows, C, 8, 16, 16, T, 0) <= min(sum(rows) * C * 2 + 4096, step) + 8 * T * 128 * 256 * 4 + 16 * T * C * 2
    for rows in ((0,), (0, 0, 0), (0, 5, 0), (5, 0)):                                 # empty pieces end the walk over the steps like others
        assert need(rows, 72, 8, 16, 1, 40) + _lib.WS_HEADER < _lib.WS_HEADER + (1 << 20)
    assert need((24, 7), 3592, 8, 16, 16, 20, 0) >= 31 * 3592 * 2                     # decode sizes with column orders go the same way


def test_mixed_stacks_decode_only_what_needs_it():
    """From 3 rows a piece of a format without a matrix-core kernel is decoded into the workspace; its neighbours' tags are read."""
    L = _lib.lib()
    mat = lambda R, C, d, bits, off: _lib.SqMatrix(0x10000, 0x20000, 0x30000, None, None, None, None, R, C, d, bits, 1, 1, (C // d * bits + 31) // 32, off)
    need = lambda mats, B, which: L.sq_workspace_bytes(_lib.matrix_array(mats), len(mats), B, which)
    for d, bits in ((8, 16), (4, 12)):
        for B in (3, 16, 32):
            large, small = mat(18944, 3584, d, bits, 0), mat(64, 3584, 8, 14, 18944)
            alone = max(need([large], B, 0), _lib.WS_HEADER), need([small], B, 0)
            assert 64 * 3584 * 2 <= alone[1] - _lib.WS_HEADER < 4 << 20
            for which in (0, 1):
                assert max(alone) <= need([large, small], B, which) < _lib.WS_HEADER + 32 * 18944 * B * 4 + (4 << 20)
                assert need([large, small], B, which) == need([small, large], B, which) == need([large, small, mat(0, 3584, d, bits, 19008)], B, which)
    assert need([mat(64, 3584, 8, 14, 0)], 2, 0) == 0
    # few short rows are through the vector kernel before a decode is: none of it is asked for
    for R, C, d, bits, rows in ((512, 1024, 4, 14, 3), (512, 1024, 4, 14, 4), (2048, 512, 4, 6, 5), (4864, 896, 4, 6, 4), (256, 520, 8, 16, 4)):
        assert need([mat(R, C, d, bits, 0)], rows, 0) == 0
    for R, C, d, bits, rows in ((512, 1024, 4, 14, 6), (16384, 512, 4, 6, 4), (4864, 896, 4, 6, 8), (256, 2080, 8, 16, 3), (5120, 2080, 8, 16, 3)):
        assert need([mat(R, C, d, bits, 0)], rows, 0) >= _lib.WS_HEADER + R * C * 2


def test_tile_gemm_waits_for_its_reads_before_the_barrier(tmp_path):
    """Behind the barrier of a slab the ring's slots are overwritten by copies that no compiler dependence ties to the reads, so
    the source itself has to wait for them: in the assembly of every variant the wait in front of a barrier behind LDS reads names
    the LDS counter."""
    import os
    import subprocess
    from quantexperiments_amd import build
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "gemm256.s"
    subprocess.run([hipcc, *build.FLAGS, "-S", "--offload-device-only", str(build.CSRC / "sq_gemm256.hip"), "-o", str(out)], check=True,
                   capture_output=True, env=dict(os.environ, TMPDIR=str(tmp_path)))
    variants = 0
    for body in re.split(r"(?m)^(?=_ZN2sq14gemm256_kernel\w+:)", out.read_text())[1:]:
        lines = [l.split(";")[0].strip() for l in body[:body.index(".Lfunc_end")].splitlines()]
        lines = [l for l in lines if l and not l.startswith(".")]
        reads, waits = False, []
        for i, l in enumerate(lines):
            reads = reads or l.startswith("ds_read")
            if l == "s_barrier" and reads:
                waits.append(next(w for w in reversed(lines[:i]) if w.startswith("s_waitcnt")))
        assert waits and all("lgkmcnt(0)" in w for w in waits), waits
        variants += 1
    assert variants == 9


def test_tile_gemm_accumulators_and_stores(tmp_path):
    """The accumulators are registers that the source names, so nothing else may live in them; and a tile's first slab does not wait
    for the 8 MT stores of the whole tile before it, so there have to be that many (as many again at a matrix' edges, 16 MT of a part's)."""
    import os
    import subprocess
    from quantexperiments_amd import build
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "gemm256.s"
    subprocess.run([hipcc, *build.FLAGS, "-S", "--offload-device-only", str(build.CSRC / "sq_gemm256.hip"), "-o", str(out)], check=True,
                   capture_output=True, env=dict(os.environ, TMPDIR=str(tmp_path)))
    variants = 0
    for body in re.split(r"(?m)^(?=_ZN2sq14gemm256_kernel\w+:)", out.read_text())[1:]:
        lines = [l.split(";")[0].strip() for l in body[:body.index(".Lfunc_end")].splitlines()]
        lines = [l for l in lines if l and not l.startswith(".")]
        assert all(l.startswith(("v_mfma_", "v_accvgpr_read")) for l in lines if re.search(r"\ba(\[\d|\d)", l))
        ep, mt = map(int, re.match(r"_ZN2sq14gemm256_kernelILi(\d)ELi(\d)E", body).groups())
        if ep:
            assert sum(l.startswith("global_store_dwordx4") for l in lines) == 32 * mt
        variants += 1
    assert variants == 9


def test_head_conversion_leaves_loads_alone(tmp_path):
    """The head kernels that convert their activations load them in an asm statement and wait for them, by count, in another: nothing
    the compiler puts anywhere may read or write the registers that these name."""
    import os
    import subprocess
    from quantexperiments_amd import build
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "q8.s"
    subprocess.run([hipcc, *build.FLAGS, "-S", "--offload-device-only", str(build.CSRC / "sq_q8.hip"), "-o", str(out)], check=True,
                   capture_output=True, env=dict(os.environ, TMPDIR=str(tmp_path)))
    variants = 0
    for body in re.split(r"(?m)^(?=_ZN2sq14q8_mfma_kernel\w+:)", out.read_text())[1:]:
        if "Lb1E" not in body.split(":", 1)[0]:
            continue
        asm, loads, takes = False, 0, 0
        for l in body[:body.index(".Lfunc_end")].splitlines():
            asm = True if "#ASMSTART" in l else False if "#ASMEND" in l else asm
            l = l.split(";")[0].strip()
            if not l or l.startswith(".") or l.endswith(":"):
                continue
            used = {r for m in re.finditer(r"\bv(?:\[(\w+)(?::(\w+))?\]|(\d+)\b)", l) for r in range(int(m[1] or m[3], 0), int(m[2] or m[1] or m[3], 0) + 1)}
            if asm and used & set(range(112, 128)):
                assert l.startswith(("global_load_dwordx4 v[", "v_mov_b32")), l
                loads, takes = loads + l.startswith("global"), takes + l.startswith("v_mov")
            else:
                assert not used & set(range(112, 128)) and not l.startswith("scratch_"), l
        assert loads and takes >= 4 * loads
        variants += 1
    assert variants == 24


def test_one_tile_gemm_waits_for_its_reads_before_the_barrier(tmp_path):
    """As for the tile kernel: the copies behind a slab's barrier overwrite slots that LDS reads may still be on their way from; and its
    accumulators, tied to written-out products, are not copied or spilled within the loop over the slabs."""
    import os
    import subprocess
    from quantexperiments_amd import build
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "gemm256.s"
    subprocess.run([hipcc, *build.FLAGS, "-S", "--offload-device-only", str(build.CSRC / "sq_gemm256.hip"), "-o", str(out)], check=True,
                   capture_output=True, env=dict(os.environ, TMPDIR=str(tmp_path)))
    variants = 0
    for body in re.split(r"(?m)^(?=_ZN2sq18gemm256_one_kernel\w+:)", out.read_text())[1:]:
        lines = [l.split(";")[0].strip() for l in body[:body.index(".Lfunc_end")].splitlines()]
        lines = [l for l in lines if l and not (l.startswith(".") and not l.startswith(".LBB"))]
        reads, waits = False, []
        for i, l in enumerate(lines):
            reads = reads or l.startswith("ds_read")
            if l == "s_barrier" and reads:
                waits.append(next(w for w in reversed(lines[:i]) if w.startswith("s_waitcnt")))
        assert waits and all("lgkmcnt(0)" in w for w in waits), waits
        first = next(i for i, l in enumerate(lines) if l.startswith("v_mfma"))
        last = max(i for i, l in enumerate(lines) if l.startswith("v_mfma"))
        assert not any(l.startswith(("v_accvgpr", "scratch_")) for l in lines[first:last])
        variants += 1
    assert variants == 9


def test_sieve_waits_for_its_codebook_slice(tmp_path):
    """Every wave gathers from the whole slice, which the waves have copied to LDS between them: in front of the first barrier the source
    has to wait for this wave's copies itself, for no barrier does.  In the assembly of every variant the wait right there leaves at most
    as many operations on their way as have been issued, on every path, behind the last copy."""
    import os
    import subprocess
    from quantexperiments_amd import build
    try:
        hipcc = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "sieve.s"
    subprocess.run([hipcc, *build.FLAGS, "-S", "--offload-device-only", str(build.CSRC / "sq_sieve.hip"), "-o", str(out)], check=True,
                   capture_output=True, env=dict(os.environ, TMPDIR=str(tmp_path)))
    variants = 0
    for body in re.split(r"(?m)^(?=_ZN2sq12sieve_kernel\w+:)", out.read_text())[1:]:
        tiles = int(re.match(r"_ZN2sq12sieve_kernelILi(\d)E", body)[1])
        lines = [l.split(";")[0].strip() for l in body[:body.index(".Lfunc_end")].splitlines()]
        lines = [l for l in lines if l and (not l.startswith(".") or l.startswith(".LBB"))]
        barrier = lines.index("s_barrier")
        copies = [i for i, l in enumerate(lines) if l.startswith("buffer_load") and l.endswith(" lds")]
        assert len(copies) == 8 and copies[-1] < barrier
        branch = next(i for i, l in enumerate(lines) if i > copies[-1] and l.startswith(("s_cbranch", ".LBB")))
        behind = sum(l.startswith(("global_load", "buffer_load", "flat_load")) for l in lines[copies[-1] + 1:branch])
        wait = re.fullmatch(r"s_waitcnt .*vmcnt\((\d+)\).*", lines[barrier - 1])
        assert wait and int(wait[1]) <= min(tiles + 1, behind), lines[barrier - 4:barrier + 1]
        variants += 1
    assert variants == 4
