"""The C-ABI library: loads, exports every symbol include/p3v.h declares, and the
ctypes signatures cover exactly that set.  No compute calls (no GPU here)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    h = open(os.path.join(ROOT, "include", "p3v.h")).read()
    h = re.sub(r"/\*.*?\*/", "", h, flags=re.S)
    return sorted(set(re.findall(r"\b(p3v_[a-z0-9_]+)\s*\(", h)))


def test_header_symbols_are_exported_and_bound():
    from phi_3_vision_mlx_amd import _lib
    assert os.path.exists(_lib.LIB_PATH), "libp3v.so not built: run __graft_entry__.build()"
    lib = ctypes.CDLL(_lib.LIB_PATH)
    syms = declared_symbols()
    assert len(syms) >= 25
    for s in syms:
        assert hasattr(lib, s), f"{s} declared in include/p3v.h but not exported by libp3v.so"
    assert sorted(_lib.SIGNATURES) == syms, set(_lib.SIGNATURES) ^ set(syms)
    assert _lib.lib().p3v_version() == 600
    assert _lib.lib().p3v_strerror(-22).decode().startswith("invalid argument")


def test_struct_layouts_match_header_field_order():
    from phi_3_vision_mlx_amd import _lib
    h = open(os.path.join(ROOT, "include", "p3v.h")).read()
    for cname, cls in (("p3v_gemm_args_t", _lib.GemmArgs), ("p3v_gemv_args_t", _lib.GemvArgs),
                       ("p3v_attn_args_t", _lib.AttnArgs), ("p3v_attn_decode_args_t", _lib.AttnDecArgs),
                       ("p3v_attn_decode_q8_args_t", _lib.AttnDecQ8Args), ("p3v_gemv_fp8_args_t", _lib.GemvF8Args)):
        end = h.index("} " + cname)
        body = h[h.rindex("typedef struct {", 0, end) + len("typedef struct {"):end]
        body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
        names = []
        for stmt in body.split(";"):
            stmt = stmt.strip()
            if not stmt:
                continue
            decl = re.sub(r"^(const\s+)?(void|uint16_t|uint8_t|uint32_t|int32_t|int64_t|float|int)\s*\*?\s*", "", stmt)
            names += [n.strip().lstrip("*").strip() for n in decl.split(",")]
        assert names == [f for f, _ in cls._fields_], (cname, names)


def test_ops_fail_loudly_without_gpu_or_library(monkeypatch):
    import pytest
    import torch
    from phi_3_vision_mlx_amd import _lib, ops
    if not torch.cuda.is_available():
        with pytest.raises(RuntimeError):
            ops.rmsnorm(torch.zeros(1, 8, dtype=torch.bfloat16), torch.zeros(8, dtype=torch.bfloat16), 1e-5)
        from phi_3_vision_mlx_amd.model import Phi3VModel
        with pytest.raises(RuntimeError):
            Phi3VModel(None, {})
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libp3v.so")
    with pytest.raises(RuntimeError, match="no CPU/PyTorch fallback"):
        _lib.lib()


def test_row_projections_check_what_they_are_given(monkeypatch):
    """gemm_merge, gemm_rows_resid, gemm_rows_scaled: a given output of another type or size, a weight of another width, too few sums of
    squares -- an error before anything is launched; what fits is launched, rows of a wider matrix among it (launches are recorded here,
    tensors are on the CPU)."""
    import types

    import torch
    from phi_3_vision_mlx_amd import _lib, ops
    real, launched, bf = _lib.lib(), [], torch.bfloat16
    stub = types.SimpleNamespace(p3v_gemm_merge_ws_bytes=real.p3v_gemm_merge_ws_bytes, p3v_gemm_rows_resid_parts=real.p3v_gemm_rows_resid_parts,
                                 **{n: lambda *a, n=n: launched.append(n) or 0 for n in ("p3v_gemm_merge", "p3v_gemm_rows_resid", "p3v_gemm_rows_scaled")})
    monkeypatch.setattr(ops.L, "lib", lambda: stub)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_chk", lambda t, dtype, name: t)
    monkeypatch.setattr(ops, "_merge_ws", {})
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)

    def rows(m, n, dtype=bf):
        return torch.empty((m, n), dtype=dtype)
    a, w, K = rows(112, 3072), rows(2 * 4096, 3072), 3072

    def merge(out):
        return ops.gemm_merge(a, w, ops.EPI_SILU_MUL, out)
    x, wo, nw, scaled, sq = rows(12, K), rows(3072, K), rows(1, 3072)[0], rows(12, 3072), rows(192, 16, torch.float32)

    def resid(out):
        return ops.gemm_rows_resid(x, wo, rows(12, 3072), nw, scaled, sq, out=out)
    wg = rows(2 * 64, K)

    def behind(out, w=wg, sq=sq, parts=192):
        return ops.gemm_rows_scaled(scaled, w, sq, parts, 1e-5, ops.EPI_SILU_MUL, out=out)
    for call, m, n in ((merge, 112, 4096), (resid, 12, 3072), (behind, 12, 64)):
        for bad in (rows(m, n, torch.float32), rows(m - 1, n), rows(m, n - 8), rows(m, n + 8), rows(m, 2 * n)[:, ::2], rows(n, m).t()):
            with pytest.raises(ValueError):
                call(bad)
        assert not launched, call
        call(rows(m, n))
        if call is not resid:                                    # (whose output lies as its residual does)
            call(rows(m, n + 8)[:, :n])
        assert launched
        launched.clear()
    for kw in (dict(w=rows(128, K + 64)), dict(w=rows(128, K - 64)), dict(sq=rows(191, 16, torch.float32)), dict(parts=193)):
        with pytest.raises(ValueError):
            behind(None, **kw)
    assert not launched
    assert behind(None).shape == (12, 64) and launched


def test_a_graphs_workspace_is_its_threads_alone(monkeypatch):
    """While one thread builds a graph in a workspace the graph owns, another thread's launches get their stream's (buffers on the CPU here)."""
    import threading

    import torch
    from phi_3_vision_mlx_amd import ops
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_gemm_ws", {})
    monkeypatch.setattr(ops, "_merge_ws", {})
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    dev, holder, other = torch.device("cpu"), {}, []

    def ask():
        return [f(dev, 8192).data_ptr() for f in (ops._gemm_workspace, ops._merge_workspace)]

    def beside():
        t = threading.Thread(target=lambda: other.append(ask()))
        t.start(), t.join()
    for frozen in (False, True):
        with ops.owned_gemm_workspace(holder, frozen=frozen):
            mine = ask()
            beside()
            assert ask() == mine == [holder["buf"].data_ptr(), holder["merge"].data_ptr()]
    assert other[0] == other[1] == ask() and not set(other[0]) & set(mine)


def test_library_never_allocates_or_reads_the_environment_per_launch():
    """include/p3v.h: launches never allocate or synchronise (callers pass workspaces, e.g. p3v_gemm_ws_bytes); knobs come
    from ONE table filled once (p3v_runtime.hip).  Checked on the sources and on the library's undefined symbols."""
    import subprocess
    csrc = os.path.join(ROOT, "phi-3-vision-mlx_amd", "csrc")
    for f in os.listdir(csrc):
        if f.endswith((".hip", ".h")):
            src = re.sub(r"//.*", "", open(os.path.join(csrc, f)).read())
            for banned in ("hipMalloc", "hipFree", "hipDeviceSynchronize", "hipStreamSynchronize", "hipMemcpy("):
                assert banned not in src, (f, banned)
            if f != "p3v_runtime.hip":
                assert "getenv" not in src, f
    from phi_3_vision_mlx_amd import _lib
    und = subprocess.run(["nm", "-D", "--undefined-only", _lib.LIB_PATH], capture_output=True, text=True, check=True).stdout
    for banned in ("hipMalloc", "hipFree", "hipDeviceSynchronize", "hipStreamSynchronize"):
        assert not re.search(rf"\b{banned}\b", und), banned


def test_tuning_table_and_gemm_workspace_size():
    from phi_3_vision_mlx_amd import _lib
    l = _lib.lib()
    v = ctypes.c_int(0)
    assert l.p3v_get_tuning(b"gemm_splitk_max_m", ctypes.byref(v)) == 0 and v.value == 1024
    assert l.p3v_set_tuning(b"no_such_knob", 1) == -22
    assert l.p3v_set_tuning(b"combine_g", 4) == 0 and l.p3v_get_tuning(b"combine_g", ctypes.byref(v)) == 0 and v.value == 4
    assert l.p3v_set_tuning(b"combine_g", -1) == 0
    # K-slice shapes: S slices of fp32 [M, N or 2N]; none elsewhere.  17 .. 256 rows: the 128 x 64-tile kernel (one workgroup per CU:
    # 48 tiles x 4 slices for down_proj, gate_up's 256 tiles in one pass); up to 1024 rows with < 256 tiles: the 128 x 128 kernel's split
    assert l.p3v_gemm_ws_bytes(128, 3072, 8192, _lib.EPI_RESID_BF16) == 4 * 128 * 3072 * 4
    assert l.p3v_gemm_ws_bytes(128, 8192, 3072, _lib.EPI_SILU_MUL) == 0
    assert l.p3v_gemm_ws_bytes(300, 3072, 8192, _lib.EPI_RESID_BF16) == 4 * 300 * 3072 * 4
    assert l.p3v_gemm_ws_bytes(2531, 3072, 8192, _lib.EPI_RESID_BF16) == 0
    assert l.p3v_gemm_ws_bytes(8, 3072, 8192, _lib.EPI_NONE) == 0
    assert l.p3v_gemm_ws_bytes(128, 3072, 8192, _lib.EPI_BIAS) == 0


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("n_split", list(range(13, 25)))
def test_fused_decode_attention_role_placement_is_a_bijection(n_split, mode):
    """p3v_attention_decode_fused_role (round 6): the 1-D grid of the fused attention + o_proj launch.  For every cache capacity
    the fused form takes (13 .. 24 tiles of 128 keys, 32 heads, o_n = 3072): every (head, split) is played by exactly one
    workgroup, every projection unit 0 .. 383 by exactly one, the 32 merging workgroups are the LAST workgroups of virtual CUs
    224 .. 255 (workgroups L, L + 256, L + 512 share a CU) and nobody on those CUs carries a projection unit; every other CU's
    last workgroup carries one (placement 2: also the second ones; placement 1: those sit on second-to-last workgroups)."""
    from phi_3_vision_mlx_amd import _lib
    l = _lib.lib()
    nh, o_n = 32, 3072
    G = nh * n_split
    out = (ctypes.c_int * 4)()
    roles = []
    for wg in range(G):
        assert l.p3v_attention_decode_fused_role(wg, nh, n_split, o_n, mode, out) == 0
        roles.append(tuple(out))
    assert sorted((r[1], r[0]) for r in roles) == [(h, s) for h in range(nh) for s in range(n_split)]
    units = [u for r in roles for u in r[2:] if u >= 0]
    assert sorted(units) == list(range(o_n // 8))
    n_on = [sum(1 for wg in range(v, G, 256)) for v in range(256)]
    for wg, (split, head, u1, u2) in enumerate(roles):
        v, slot = wg % 256, wg // 256
        last = slot == n_on[v] - 1
        if split == n_split - 1:
            assert v == 224 + head and last and u1 < 0 and u2 < 0
        if v >= 224:
            assert u1 < 0 and u2 < 0
        elif last:
            assert u1 == v
        if mode == 2:
            assert (u1 >= 0) == (last and v < 224) and (u2 < 0 or u1 >= 0)
        else:
            assert u2 < 0 and (u1 < 0 or slot >= n_on[v] - 2)
    assert l.p3v_attention_decode_fused_role(0, 32, 12, o_n, mode, out) == _lib.ERR_UNSUPPORTED      # too few workgroups for 384 units
    assert l.p3v_attention_decode_fused_role(0, 8, 16, o_n, mode, out) == _lib.ERR_UNSUPPORTED       # not the 32-head geometry
    assert l.p3v_attention_decode_fused_role(G, nh, n_split, o_n, mode, out) == -22


@pytest.mark.parametrize("tile", [1, 4, 40, 53, 62, 73, 80, 82, 94, 99, 164, 163, 844, -84])
def test_a_pinned_gemm_tile_that_does_not_exist_is_refused(tile):
    """The knob "gemm_tile" takes any number: one that names no tile of the large GEMM kernels (or, gated, the 192-column ones) is an
    error code, not a division by zero and not another tile.  Negative: no pin.  A process of its own, since the fault would end it."""
    import subprocess
    import sys
    code = f"""
import ctypes as C
from phi_3_vision_mlx_amd import _lib as L, ops
l, buf = L.lib(), C.create_string_buffer(4096)
p = (C.addressof(buf) + 15) // 16 * 16
def gemm(M, epilogue):
    return l.p3v_gemm(C.byref(L.GemmArgs(p, p, p, 0, 0, 0, M, 768, 64, 64, 64, 768, epilogue, 0, 0, 0, 0)), None)
for t, M in (({tile}, 64), (43, 64), (63, 64), (83, 64)):
    assert l.p3v_set_tuning(b"gemm_tile", t) == 0
    if t < 0:
        assert gemm(0, ops.EPI_NONE) == 0
    elif t not in (43, 63, 83):
        assert gemm(M, ops.EPI_NONE) == L.ERR_UNSUPPORTED, (t, gemm(M, ops.EPI_NONE))
    if t > 0:
        assert gemm(M, ops.EPI_SILU_MUL) == L.ERR_UNSUPPORTED and gemm(M, ops.EPI_GELU_MUL) == L.ERR_UNSUPPORTED, t
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stderr[-1500:])


def test_k_slices_decline_partials_beyond_32_bit_offsets():
    """The partials are stored at 32-bit byte offsets from a wave's first output: 80 rows of N floats have to stay below 2^31.  (Nothing is launched.)"""
    from phi_3_vision_mlx_amd import _lib as L, ops
    l, buf, v = L.lib(), ctypes.create_string_buffer(4096), ctypes.c_int()
    p, N = (ctypes.addressof(buf) + 15) // 16 * 16, (2 ** 31 // 320 // 256 + 1) * 256
    assert l.p3v_get_tuning(b"gemm_slices", ctypes.byref(v)) == 0
    try:
        for tile in (154, 144):                                   # one slice on tiles of 160 / 128 x 256
            assert l.p3v_set_tuning(b"gemm_slices", tile) == 0
            a = L.GemmArgs(p, p, p, 0, p, 0, 1, N, 64, 64, 64, N, ops.EPI_RESID_BF16, 0, p, N * 4, 0)
            assert l.p3v_gemm_slices(ctypes.byref(a), None, 0.0, None, None) == L.ERR_UNSUPPORTED
    finally:
        l.p3v_set_tuning(b"gemm_slices", v.value)


def test_which_tile_the_plan_by_rounds_names():
    """p3v_gemm_plan (what p3v_gemm departs from only for 2 %): one size for every tile, and sizes that stay on the row packing: where no tile
    promises enough, 224-row tiles for one full round (by the plan slower than 256 x 256 there), short K loops, few rows."""
    from phi_3_vision_mlx_amd import _lib, ops
    l, v = _lib.lib(), ctypes.c_int()
    assert l.p3v_get_tuning(b"gemm_big_rows", ctypes.byref(v)) == 0 and l.p3v_set_tuning(b"gemm_big_rows", -1) == 0
    try:
        for M, N, K, epi, want in ((2531, 3072, 8192, ops.EPI_RESID_BF16, 44), (640, 8192, 3072, ops.EPI_SILU_MUL, 54), (1300, 3072, 3072, ops.EPI_NONE, 43),
                                   (900, 8192, 3072, ops.EPI_SILU_MUL, 84), (700, 8192, 3072, ops.EPI_GELU_MUL, 74), (1237, 9216, 3072, ops.EPI_NONE, 83),
                                   (2885, 4096, 1024, ops.EPI_BIAS_QGELU, 74), (9809, 1024, 4096, ops.EPI_BIAS_RESID_F32, 54),
                                   (1500, 9216, 3072, ops.EPI_NONE, 0), (1024, 9472, 3072, ops.EPI_NONE, 0), (1300, 8192, 3072, ops.EPI_SILU_MUL, 0),
                                   (2531, 3072, 512, ops.EPI_NONE, 0), (256, 8192, 3072, ops.EPI_NONE, 0), (2531, 3000, 3072, ops.EPI_NONE, 0),
                                   (2531, 1024, 1024, ops.EPI_PATCH, 0), (0, 3072, 3072, ops.EPI_NONE, 0), (2531, 3072, 3072, 99, 0)):
            assert l.p3v_gemm_plan(M, N, K, epi) == want, (M, N, K, epi, l.p3v_gemm_plan(M, N, K, epi))
    finally:
        l.p3v_set_tuning(b"gemm_big_rows", v.value)


def test_which_tile_p3v_gemm_runs():
    """The tile by how full the chip's rounds are: those of 192 rows and the other heights where they were measured the fastest, the plan's own
    answer elsewhere, and 0 for what other kernels take (few rows, K slices up to 1024 rows, short K, columns that no tile divides, a K that p3v_gemm refuses)."""
    from phi_3_vision_mlx_amd import _lib, ops
    l, v = _lib.lib(), ctypes.c_int()
    assert l.p3v_get_tuning(b"gemm_big_rows", ctypes.byref(v)) == 0 and l.p3v_set_tuning(b"gemm_big_rows", -1) == 0
    try:
        for M, N, K, epi, want in ((768, 8192, 3072, ops.EPI_SILU_MUL, 64), (2300, 8192, 3072, ops.EPI_SILU_MUL, 64), (2531, 8192, 3072, ops.EPI_SILU_MUL, 74),
                                   (2531, 9216, 3072, ops.EPI_NONE, 64), (900, 9216, 3072, ops.EPI_NONE, 63), (6000, 3072, 8192, ops.EPI_RESID_BF16, 63),
                                   (8192, 3072, 8192, ops.EPI_RESID_BF16, 83), (9809, 4096, 1024, ops.EPI_BIAS_QGELU, 74), (640, 8192, 3072, ops.EPI_SILU_MUL, 54),
                                   (300, 3072, 3072, ops.EPI_NONE, 0), (500, 3072, 8192, ops.EPI_RESID_BF16, 0), (300, 3072, 3072, ops.EPI_BIAS, 43), (128, 8192, 3072, ops.EPI_SILU_MUL, 0),
                                   (2531, 3072, 3080, ops.EPI_NONE, 0),
                                   (2531, 3072, 512, ops.EPI_NONE, 0), (256, 8192, 3072, ops.EPI_NONE, 0), (2531, 3000, 3072, ops.EPI_NONE, 0), (0, 3072, 3072, ops.EPI_NONE, 0)):
            assert (l.p3v_gemm_ws_bytes(M, N, K, epi) > 0) <= (want == 0)
            assert l.p3v_gemm_tile(M, N, K, epi) == want, (M, N, K, epi, l.p3v_gemm_tile(M, N, K, epi))
    finally:
        l.p3v_set_tuning(b"gemm_big_rows", v.value)


def test_which_tile_runs_an_fp8_projection():
    """A pin names the tile that runs, for odd numbers of K-tiles too; one that the problem does not divide into leaves the choice by shape."""
    from phi_3_vision_mlx_amd import _lib, ops
    l, v = _lib.lib(), ctypes.c_int()
    assert l.p3v_get_tuning(b"gemm_f8_narrow", ctypes.byref(v)) == 0
    try:
        for K in (256, 384, 640, 3200):
            for tile in (44, 54, 42, 43, 64, 74, 84, 32, 22, 21, 11):
                assert l.p3v_set_tuning(b"gemm_f8_narrow", tile) == 0
                assert l.p3v_gemm_fp8_tile(1300, 9216, K, ops.EPI_NONE) == tile, (K, tile)
                if tile % 2 == 0:
                    assert l.p3v_gemm_fp8_tile(1300, 8192, K, ops.EPI_SILU_MUL) == tile, (K, tile)
        assert l.p3v_set_tuning(b"gemm_f8_narrow", 43) == 0
        free = l.p3v_gemm_fp8_tile(1300, 4096, 384, ops.EPI_NONE)
        assert free != 43 and l.p3v_set_tuning(b"gemm_f8_narrow", -1) == 0 and l.p3v_gemm_fp8_tile(1300, 4096, 384, ops.EPI_NONE) == free
        # (by shape: the fastest measured tile, by 5 % or more, of short K, of K = 3072 and 8192, of odd numbers of K-tiles)
        for M, N, K, epi, want in ((1300, 4096, 384, ops.EPI_NONE, 44), (768, 9216, 640, ops.EPI_NONE, 44), (1300, 9216, 640, ops.EPI_NONE, 64), (1300, 9216, 3200, ops.EPI_NONE, 64),
                                   (1024, 9216, 3072, ops.EPI_NONE, 54), (320, 9216, 3072, ops.EPI_NONE, 42), (2531, 9216, 3072, ops.EPI_NONE, 64),
                                   (2531, 8192, 3072, ops.EPI_SILU_MUL, 74), (2048, 8192, 2944, ops.EPI_SILU_MUL, 84), (2531, 3072, 8192, ops.EPI_RESID_BF16, 44),
                                   (4096, 3072, 3072, ops.EPI_RESID_BF16, 74),
                                   (137, 3072, 8192, ops.EPI_RESID_BF16, 11), (276, 3072, 8192, ops.EPI_RESID_BF16, 21), (512, 3072, 8192, ops.EPI_RESID_BF16, 22),
                                   (803, 3072, 8192, ops.EPI_RESID_BF16, 32), (137, 3072, 3072, ops.EPI_RESID_BF16, 11), (137, 9216, 3072, ops.EPI_NONE, 22),
                                   (276, 9216, 3072, ops.EPI_NONE, 32), (128, 8192, 3072, ops.EPI_SILU_MUL, 22), (257, 8192, 3072, ops.EPI_SILU_MUL, 44)):
            assert l.p3v_gemm_fp8_tile(M, N, K, epi) == want, (M, N, K, epi, l.p3v_gemm_fp8_tile(M, N, K, epi))
        for M, n_q, n_kv, K, want in ((256, 3072, 3072, 3072, 0), (577, 3072, 3072, 3072, 1), (768, 3072, 3072, 3072, 1), (1024, 3072, 3072, 3072, 0), (1800, 3072, 3072, 3072, 0), (2048, 3072, 3072, 3072, 0),
                                      (2531, 3072, 3072, 3072, 1), (2700, 3072, 3072, 3072, 0), (4096, 3072, 3072, 3072, 1), (6000, 3072, 3072, 3072, 1), (8192, 3072, 3072, 3072, 1), (16384, 3072, 3072, 3072, 1), (2531, 1024, 1024, 1024, 1), (1536, 768, 768, 384, 1)):
            assert l.p3v_gemm_qkv_fp8_pays(M, n_q, n_kv, K) == want, (M, n_q, n_kv, K)
        # (in front of p3v_rope_kv_quantize: the faster side of whole prompts run either way, by 5 us a layer or more)
        for M, want in ((137, 0), (276, 0), (803, 0), (1024, 0), (1800, 0), (2300, 0), (2700, 0), (3300, 0), (3900, 0), (4050, 1), (4096, 1), (4500, 0), (4700, 0), (5200, 1),
                        (6500, 0), (7300, 0), (7600, 0), (7800, 0), (8000, 1), (8192, 0), (10000, 0), (65536, 0), (0, 0)):
            assert l.p3v_gemm_qkv_fp8_stored_pays(M, 3072, 3072, 3072) == want, M
        assert l.p3v_gemm_qkv_fp8_stored_pays(4096, 3000, 3072, 3072) == 0
        for M, N, K, epi in ((0, 256, 256, ops.EPI_NONE), (1, 100, 256, ops.EPI_NONE), (1, 256, 64, ops.EPI_NONE), (1, 256, 256, ops.EPI_GELU_MUL)):
            assert l.p3v_gemm_fp8_tile(M, N, K, epi) == 0
    finally:
        l.p3v_set_tuning(b"gemm_f8_narrow", v.value)


def test_which_projections_pay_in_one_pass_and_which_ask_for_more_slices():
    """p3v_gemm_one_pass_pays: 257 .. 384 rows, more than 128 and at most 256 tiles of 128 x 128, where K slices would run otherwise.  p3v_gemm_ws_most_bytes: up to 256 rows,
    whole 96 columns, slices of 12 K-tiles, 16 beyond 128 rows; p3v_gemm_ws_bytes where the kernel for 9 .. 32 rows or another takes the shape."""
    from phi_3_vision_mlx_amd import _lib, ops
    l = _lib.lib()
    for M, tiles, K, epi, want in ((300, 42, 3072, ops.EPI_NONE, 0), (300, 43, 3072, ops.EPI_NONE, 1), (300, 85, 3072, ops.EPI_NONE, 1), (300, 86, 3072, ops.EPI_NONE, 0),
                                   (256, 72, 3072, ops.EPI_NONE, 0), (257, 72, 3072, ops.EPI_NONE, 1), (384, 72, 512, ops.EPI_NONE, 1), (385, 72, 3072, ops.EPI_NONE, 0),
                                   (300, 72, 3072, ops.EPI_RESID_BF16, 0), (300, 72.5, 3072, ops.EPI_NONE, 0), (300, 72, 3136, ops.EPI_NONE, 0), (0, 72, 3072, ops.EPI_NONE, 0)):
        assert l.p3v_gemm_one_pass_pays(M, int(tiles * 128), K, epi) == want, (M, tiles, K, epi)
    for M, N, K, few, most in ((9, 3072, 8192, 4, 4), (32, 3072, 8192, 4, 4), (20, 3072, 6144, 4, 8), (33, 3072, 8192, 4, 8), (128, 3072, 6144, 4, 8), (129, 3072, 8192, 2, 4),
                               (256, 3072, 8192, 2, 4), (257, 3072, 8192, 4, 4), (200, 3072, 4096, 2, 4), (100, 3072, 4096, 4, 4), (200, 3072, 3072, 2, 2), (128, 3000, 8192, 0, 0)):
        got = [f(M, N, K, ops.EPI_RESID_BF16) / (4 * M * N) for f in (l.p3v_gemm_ws_bytes, l.p3v_gemm_ws_most_bytes)]
        assert got == [few, most], (M, N, K, got)


def test_which_tile_runs_a_qkv_projection():
    """From 1024 rows on the fastest measured tile of (rows, rows of W for Q, for K and V, K): 128 x 128 ones at short K, every height at the decoder's
    widths and the vision tower's; the knob names the same numbers; other regions, few rows and odd K are not priced."""
    from phi_3_vision_mlx_amd import _lib
    l, v, r = _lib.lib(), ctypes.c_int(), ctypes.c_int()
    assert l.p3v_get_tuning(b"gemm_qkv_flat", ctypes.byref(v)) == 0 and l.p3v_get_tuning(b"gemm_big_rows", ctypes.byref(r)) == 0 and l.p3v_set_tuning(b"gemm_big_rows", -1) == 0
    try:
        for args, want in (((1536, 1536, 1536, 512), 1), ((8192, 1536, 1536, 512), 1), ((6000, 3072, 3072, 768), 1), ((1024, 1024, 1024, 256), 1), ((1154, 1024, 1024, 1024), 2),
                           ((1536, 3072, 3072, 3072), 7), ((2048, 3072, 3072, 3072), 5), ((4096, 3072, 3072, 3072), 7), ((2531, 3072, 3072, 3072), 6), ((16384, 3072, 3072, 3072), 8),
                           ((2885, 1024, 1024, 1024), 5), ((900, 3072, 3072, 3072), 5), ((2531, 3072, 3072, 100), 0), ((2531, 3072, 384, 3072), 0), ((256, 3072, 3072, 3072), 0), ((0, 3072, 3072, 3072), 0)):
            assert l.p3v_set_tuning(b"gemm_qkv_flat", -1) == 0
            assert l.p3v_gemm_qkv_tile(*args) == want, (args, l.p3v_gemm_qkv_tile(*args))
            if want and args[0] >= 1024:
                for pin in (1, 4, 8):
                    assert l.p3v_set_tuning(b"gemm_qkv_flat", pin) == 0 and l.p3v_gemm_qkv_tile(*args) == pin
    finally:
        l.p3v_set_tuning(b"gemm_qkv_flat", v.value), l.p3v_set_tuning(b"gemm_big_rows", r.value)


def test_which_decode_batches_run_one_workgroup_per_row_and_head():
    """(rows, new tokens, heads, kv heads, capacity) where the form was measured faster, and where it was not: an uneven second round
    of pairs, shared kv heads, few pairs, long caches."""
    from phi_3_vision_mlx_amd import _lib
    fit = _lib.lib().p3v_attention_decode_rows_fit
    for yes in ((4, 1, 32, 32, 128), (4, 1, 32, 32, 192), (8, 1, 32, 32, 192), (12, 1, 32, 32, 192), (16, 1, 32, 32, 256), (9, 1, 32, 32, 256), (9, 4, 32, 32, 192),
                (15, 1, 32, 32, 640), (6, 1, 32, 32, 512), (8, 1, 32, 8, 256), (9, 1, 32, 8, 128), (14, 1, 32, 8, 192), (16, 16, 32, 32, 256), (32, 1, 16, 16, 192)):
        assert fit(*yes) == 1, yes
    for no in ((9, 1, 32, 32, 192), (10, 1, 32, 32, 192), (11, 1, 32, 32, 192), (4, 1, 32, 8, 256), (6, 1, 32, 8, 256), (9, 1, 32, 8, 192), (9, 1, 32, 8, 256), (12, 1, 32, 8, 192),
               (12, 1, 32, 32, 576), (4, 1, 32, 32, 320), (3, 1, 32, 32, 128), (17, 1, 32, 32, 128), (8, 1, 32, 32, 704), (0, 1, 32, 32, 128), (4, 1, 32, 0, 128), (4, 1, 32, 5, 128)):
        assert fit(*no) == 0, no


@pytest.mark.parametrize("B,T,n_split", [(1, 6272, 49), (1, 16384, 128), (1, 16512, 40), (8, 2688, 21), (16, 16256, 127), (32, 8064, 63), (32, 8192, 64), (64, 4096, 32), (64, 4224, 1),
                                         (32, 8320, 2), (64, 16256, 1), (512, 640, 1)])
def test_how_many_workgroups_attend_an_int8_cache(monkeypatch, B, T, n_split):
    """A 128-key tile a workgroup as far as that was measured, 65536 workgroups and their partials; the walking kernel's few splits beyond, however many rows."""
    from types import SimpleNamespace
    from phi_3_vision_mlx_amd import model, ops
    monkeypatch.delenv("P3V_ATTN_NSPLIT", raising=False), monkeypatch.delenv("P3V_ATTN_TILE128", raising=False)
    monkeypatch.setattr(ops, "attention_ws", lambda B, L, nh, hd, n, dev: ops.attention_ws_bytes(B, L, nh, hd, n))
    bufs = {}
    model.Phi3VModel._split_plan(SimpleNamespace(cfg=SimpleNamespace(num_attention_heads=32), hd=96, device="cpu"), bufs, B, 1, T, quantized=True)
    assert bufs["n_split"] == n_split and bufs["ws"] <= 65536 * 16 * 98 * 4


@pytest.mark.parametrize("held", ["bf16", "q4", "fp8"])
def test_which_prompt_projections_ask_for_the_most_slices(monkeypatch, held):
    """Weights that lie in memory: up to 256 rows; weights expanded into the scratch in front of the product: 129 .. 256."""
    from types import SimpleNamespace
    import torch
    from phi_3_vision_mlx_amd import model, ops
    seen, w = [], torch.empty((3072, 8192), dtype=torch.bfloat16, device="meta")
    monkeypatch.setattr(ops, "gemm", lambda *a, **k: seen.append(("gemm", k["slices"])))
    monkeypatch.setattr(ops, "gemm_slices", lambda *a, **k: seen.append(("slices", k["few_rows"])))
    for f in ("dequant_q4", "dequant_fp8"):
        monkeypatch.setattr(ops, f, lambda *a, **k: w)
    me = SimpleNamespace(cfg=SimpleNamespace(rms_norm_eps=1e-5), fp8_act=False, serving=False, w={"k": w}, _deq=torch.empty(3072 * 8192, device="meta"),
                         w8={"k": (w, None)} if held == "fp8" else {}, w4={"k": (torch.empty((3072, 1024), device="meta"), None)} if held == "q4" else {})
    for M in (33, 128, 129, 256, 257):
        most = M <= 256 and (M > 128 or held == "bf16")
        for epi in (ops.EPI_NONE, ops.EPI_RESID_BF16):
            seen.clear()
            x = torch.empty((M, 8192), device="meta")
            model.Phi3VModel._proj_frozen(me, x, "k", epi, resid=x, out=x)
            assert seen == ([("slices", most)] if epi == ops.EPI_RESID_BF16 else []) + [("gemm", "most" if most else True)], (M, epi, seen)


def test_fused_qkv_projections_decline_several_rows_of_fewer_than_seven_tokens():
    """The V^T epilogue's runs of eight tokens cross the end of one batch row at most.  Everything else about these calls is taken, so
    the answer comes from that check (no kernel starts: declined on the host)."""
    from phi_3_vision_mlx_amd import _lib as L, ops
    l = L.lib()
    buf = ctypes.create_string_buffer(4096)
    p = (ctypes.addressof(buf) + 15) // 16 * 16
    hd, nh, K = 64, 16, 128
    N = 3 * nh * hd
    for B, Lq in ((5, 3), (30, 6), (2, 1), (300, 4), (180, 6)):
        M = B * Lq
        sp = L.QkvSplit(0, 0, p, p, p, B, Lq, nh, nh, hd, 0, 128, 1, 0, 1, 1.0)
        assert l.p3v_gemm_qkv(ctypes.byref(L.GemmArgs(p, p, 0, 0, 0, 0, M, N, K, K, K, N, ops.EPI_NONE, 0, 0, 0, 0)), ctypes.byref(sp), None) == L.ERR_UNSUPPORTED
        assert l.p3v_gemm_qkv_fp8(ctypes.byref(L.GemmF8Args(p, p, p, p, 0, 0, M, N, K, K, K, N, ops.EPI_NONE)), ctypes.byref(sp), None) == L.ERR_UNSUPPORTED


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "phi-3-vision-mlx_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                src = open(os.path.join(dirpath, f)).read()
                assert "phi3v_oracle" not in src and "import oracle" not in src and "from oracle" not in src, f


@pytest.mark.skipif(os.environ.get("P3V_ASAN") != "1", reason="opt-in (P3V_ASAN=1): a ~50 s AddressSanitizer host build of libp3v.so")
def test_asan_host_build_of_the_launchers():
    """`-fsanitize=address` HOST build of the extension; its launchers' argument validation, workspace
    sizing and tuning table are driven without a GPU (tools/asan_host_check.cpp).  profiles/r04_asan_host_check.txt holds a run."""
    import subprocess
    r = subprocess.run(["bash", os.path.join(ROOT, "tools", "asan_host_build.sh")], capture_output=True, text=True, timeout=1200)
    assert r.returncode == 0 and "all launcher argument paths clean" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
