"""CPU-only checks of the host side: the Python surface mirrors the reference's, every
validation rule raises before the device is touched, the C-ABI library loads and
exports what include/grouped_gemm_hip.h declares, and the golden fixture of
configuration 1 still matches the oracle.  No GPU, no compute calls."""
import ctypes
import importlib.util
import inspect
import os
import re
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_LIB = os.path.join(ROOT, "grouped_gemm_amd", "libgrouped_gemm_hip.so")


def bf16(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


# ------------------------------------------------------------------ Python surface

def test_extension_module_imports_top_level_first():
    # setup.py:35 of the reference installs the extension under the top-level name
    # grouped_gemm_backend; here it resolves once either package has been imported, whichever
    # comes first, and torch before it (backend.py:1-3)
    import subprocess
    import sys
    for pkg in ("grouped_gemm", "grouped_gemm_amd"):
        code = (f"import sys; sys.path.insert(0, {ROOT!r}); import {pkg}; import grouped_gemm_backend as m; "
                "assert callable(m.gmm)")
        subprocess.run([sys.executable, "-c", code], check=True)


def test_package_layout_matches_reference():
    # grouped_gemm/__init__.py:1-2, ops.py:1, ops_test.py:5,154
    import grouped_gemm
    from grouped_gemm import ops
    import grouped_gemm.backend as be
    import grouped_gemm_backend
    assert ops.backend is be
    assert be.backend is grouped_gemm_backend
    assert list(inspect.signature(ops.gmm).parameters) == ["a", "b", "batch_sizes", "trans_b"]
    assert list(inspect.signature(be.gmm).parameters) == ["a", "b", "batch_sizes", "trans_a", "trans_b", "c"]
    assert inspect.signature(be.gmm).parameters["c"].default is None
    assert issubclass(ops.GroupedGemm, torch.autograd.Function)


def test_allocate_output_shapes_and_asserts():
    # grouped_gemm/backend.py:11-22
    from grouped_gemm_amd.backend import _allocate_output
    bs = torch.tensor([3, 5])
    assert _allocate_output(bf16(8, 16), bf16(2, 16, 24), bs, False, False).shape == (8, 24)
    assert _allocate_output(bf16(8, 16), bf16(2, 24, 16), bs, False, True).shape == (8, 24)
    out = _allocate_output(bf16(8, 16), bf16(8, 24), bs, True, False)
    assert out.shape == (2, 16, 24) and out.dtype == torch.bfloat16
    with pytest.raises(AssertionError):
        _allocate_output(bf16(8, 16), bf16(8, 24), bs, True, True)
    with pytest.raises(AssertionError):
        _allocate_output(bf16(8, 16), bf16(2, 16, 24), bs.view(1, 2), False, False)
    with pytest.raises(AssertionError):
        _allocate_output(bf16(2, 4, 16), bf16(2, 16, 24), bs, False, False)
    with pytest.raises(AssertionError):
        _allocate_output(bf16(8, 16), bf16(16, 24), bs, False, False)
    with pytest.raises(AssertionError):
        _allocate_output(bf16(8, 16), bf16(2, 8, 24), bs, True, False)


def test_cpu_tensors_are_rejected_by_gmm():
    # csrc/grouped_gemm.cu:490: a must be on the GPU; surfaces as RuntimeError
    from grouped_gemm import ops
    with pytest.raises(RuntimeError, match="GPU tensor"):
        ops.gmm(bf16(8, 16), bf16(2, 16, 24), torch.tensor([3, 5]))


GOOD = dict(a=(8, 16), b=(2, 16, 24), c=(8, 24), bs=[3, 5], ta=False, tb=False)


def _validate(**kw):
    import grouped_gemm_backend
    cfg = dict(GOOD)
    cfg.update(kw)
    a = cfg.get("a_t", bf16(*cfg["a"]))
    b = cfg.get("b_t", bf16(*cfg["b"]))
    c = cfg.get("c_t", bf16(*cfg["c"]))
    bs = cfg.get("bs_t", torch.tensor(cfg["bs"], dtype=torch.int64))
    grouped_gemm_backend.validate(a, b, c, bs, cfg["ta"], cfg["tb"])


def test_validate_accepts_the_three_layouts():
    _validate()
    _validate(b=(2, 24, 16), tb=True)
    _validate(b=(8, 24), c=(2, 16, 24), ta=True)


@pytest.mark.parametrize("kw", [
    dict(ta=True, tb=True),                                     # grouped_gemm.cu:476
    dict(bs_t=torch.tensor([[3, 5]])),                          # :485
    dict(bs_t=torch.tensor([3, 5], dtype=torch.int32)),         # :486
    dict(a=(2, 4, 16)),                                         # :491
    dict(a_t=torch.zeros(8, 16)),                               # :492
    dict(b_t=torch.zeros(2, 16, 24, dtype=torch.float16)),      # :505
    dict(c_t=torch.zeros(8, 24)),                               # :506
    dict(ta=True, b=(2, 4, 24), c=(2, 16, 24)),                 # :517
    dict(ta=True, b=(8, 24), c=(2 * 16, 24)),                   # :518
    dict(ta=True, b=(7, 24), c=(2, 16, 24)),                    # :519
    dict(ta=True, b=(8, 24), c=(3, 16, 24)),                    # :520
    dict(ta=True, b=(8, 24), c=(2, 8, 24)),                     # :521
    dict(ta=True, b=(8, 24), c=(2, 16, 32)),                    # :522
    dict(b=(16, 24)),                                           # :524
    dict(c=(2, 4, 24)),                                         # :525
    dict(b=(2, 8, 24)),                                         # :531 contraction mismatch
    dict(tb=True),                                              # :531 with trans_b: b.size(2) != a.size(1)
    dict(bs=[3, 4, 1]),                                         # :534
    dict(c=(8, 32)),                                            # output shape (checked here, not in the reference)
    dict(a_t=bf16(16, 8).t()),                                  # :538
    dict(b_t=bf16(2, 24, 16).transpose(1, 2)),                  # :539
    dict(c_t=bf16(24, 8).t()),                                  # :540
])
def test_validate_rejects(kw):
    with pytest.raises(RuntimeError):
        _validate(**kw)


# ------------------------------------------------------------------------ C ABI

def _declared_functions():
    text = open(os.path.join(ROOT, "include", "grouped_gemm_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(gg_[a-z0-9_]+)\s*\(", text)))


def test_c_abi_exports_every_declared_symbol():
    names = _declared_functions()
    assert {"gg_gmm_bf16", "gg_gmm", "gg_gmm_no_alloc", "gg_init", "gg_gmm_bf16_acc_f32", "gg_debug_schedule",
            "gg_last_error", "gg_version", "gg_tile_shape"} <= set(names)
    lib = ctypes.CDLL(HIP_LIB)
    for n in names:
        assert hasattr(lib, n), n


def test_c_abi_argument_errors_need_no_device():
    lib = ctypes.CDLL(HIP_LIB)
    lib.gg_last_error.restype = ctypes.c_char_p
    i64 = ctypes.c_int64
    sizes = (i64 * 2)(3, 5)
    call = lambda hin, hout, ta, tb, tokens=8, e=2: lib.gg_gmm_bf16(
        None, None, None, sizes, 0, i64(e), i64(tokens), i64(hin), i64(hout), ta, tb, None)
    assert call(16, 24, 1, 1) == -1 and b"both" in lib.gg_last_error()
    assert call(-8, 24, 0, 0) == -1
    assert call(16, 24, 0, 0, tokens=1 << 31) == -2
    assert call(16, 24, 0, 0, e=0) == 0                       # nothing to do
    # fake, never dereferenced pointers: the alignment check comes before any device call
    ptr = ctypes.c_void_p
    misaligned = lib.gg_gmm_bf16(ptr(4096), ptr(8192 + 1), ptr(12288), sizes, 0, i64(2), i64(8), i64(16),
                                 i64(24), 0, 0, None)
    assert misaligned == -2 and b"aligned to their element size" in lib.gg_last_error()
    # the accumulating form: tighter limit on the hidden sizes, checked before anything else
    acc = lib.gg_gmm_bf16_acc_f32(ptr(4096), ptr(8192), ptr(12288), sizes, 0, i64(2), i64(8), i64(1 << 20),
                                  i64(24), None)
    assert acc == -2 and b"2^20" in lib.gg_last_error()
    # host-resident sizes that would wrap a running sum are rejected one by one, before any device call
    huge = (i64 * 2)(10, (1 << 63) - 1)
    rc = lib.gg_gmm_bf16(ptr(4096), ptr(8192), ptr(12288), huge, 0, i64(2), i64(16), i64(16), i64(24), 0, 0, None)
    assert rc == -1 and b"sum past" in lib.gg_last_error()
    bm, bn, bk = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert lib.gg_tile_shape(i64(8), i64(32768), 0, 0, ctypes.byref(bm), ctypes.byref(bn), ctypes.byref(bk)) == 0
    assert (bm.value, bn.value, bk.value) == (256, 256, 64)
    assert lib.gg_tile_shape(i64(256), i64(25600), 0, 1, ctypes.byref(bm), ctypes.byref(bn), ctypes.byref(bk)) == 0
    assert bm.value == 128          # few rows per group: the shorter tile
    assert bm.value > 0 and bn.value > 0 and bk.value > 0
    assert lib.gg_version() >= 100


def test_validate_element_types():
    # past the reference (bfloat16 only, grouped_gemm.cu:492, 505-506): float16 for all three
    # tensors alike; float8 operands with a bfloat16 output
    _validate(a_t=torch.zeros(8, 16, dtype=torch.float16), b_t=torch.zeros(2, 16, 24, dtype=torch.float16),
              c_t=torch.zeros(8, 24, dtype=torch.float16))
    for f8 in (torch.float8_e4m3fn, torch.float8_e5m2):
        _validate(a_t=torch.zeros(8, 16, dtype=f8), b_t=torch.zeros(2, 16, 24, dtype=f8))     # c bfloat16
        with pytest.raises(RuntimeError):
            _validate(a_t=torch.zeros(8, 16, dtype=f8), b_t=torch.zeros(2, 16, 24, dtype=f8),
                      c_t=torch.zeros(8, 24, dtype=f8))
    with pytest.raises(RuntimeError):
        _validate(a_t=torch.zeros(8, 16, dtype=torch.float16), b_t=torch.zeros(2, 16, 24, dtype=torch.float16))
    with pytest.raises(RuntimeError):
        _validate(a_t=torch.zeros(8, 16, dtype=torch.float8_e4m3fn), b_t=torch.zeros(2, 16, 24, dtype=torch.float8_e5m2))


class _Args(ctypes.Structure):
    """gg_gmm_args of include/grouped_gemm_hip.h."""
    _fields_ = [("struct_bytes", ctypes.c_uint32), ("dtype", ctypes.c_int32),
                ("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("c", ctypes.c_void_p),
                ("batch_sizes", ctypes.c_void_p), ("batch_sizes_on_device", ctypes.c_int32),
                ("trans_a", ctypes.c_int32), ("trans_b", ctypes.c_int32), ("accumulate_f32", ctypes.c_int32),
                ("num_groups", ctypes.c_int64), ("tokens", ctypes.c_int64),
                ("hidden_in", ctypes.c_int64), ("hidden_out", ctypes.c_int64),
                ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_uint64),
                ("flags", ctypes.c_int32), ("reserved0", ctypes.c_int32), ("stream", ctypes.c_void_p),
                ("a_row_index", ctypes.c_void_p), ("b_row_index", ctypes.c_void_p), ("c_row_index", ctypes.c_void_p),
                ("a_num_rows", ctypes.c_int64), ("c_num_rows", ctypes.c_int64),
                ("epilogue", ctypes.c_int32), ("b_num_rows", ctypes.c_int32), ("size_status", ctypes.c_void_p)]


def test_general_entry_point_argument_errors_need_no_device():
    lib = ctypes.CDLL(HIP_LIB)
    lib.gg_last_error.restype = ctypes.c_char_p
    lib.gg_gmm.argtypes = [ctypes.c_void_p]
    sizes = (ctypes.c_int64 * 2)(3, 5)

    def call(**kw):
        g = _Args()
        g.struct_bytes = ctypes.sizeof(_Args)
        g.a, g.b, g.c = 4096, 8192, 12288            # never dereferenced: every case fails before the device
        g.batch_sizes = ctypes.addressof(sizes)
        g.num_groups, g.tokens, g.hidden_in, g.hidden_out = 2, 8, 16, 24
        for k, v in kw.items():
            setattr(g, k, v)
        return lib.gg_gmm(ctypes.byref(g)), lib.gg_last_error()

    assert call(struct_bytes=8)[0] == -1
    assert lib.gg_gmm(None) == -1
    assert call(dtype=9) == (-1, b"dtype must be one of GG_DTYPE_*")
    assert call(epilogue=7)[0] == -1
    rc, msg = call(epilogue=1, trans_a=1)
    assert rc == -1 and b"SwiGLU" in msg
    rc, msg = call(accumulate_f32=1)
    assert rc == -1 and b"trans_a" in msg
    rc, msg = call(trans_a=1, c_row_index=64)
    assert rc == -1 and b"c_row_index" in msg
    rc, msg = call(b_row_index=64)
    assert rc == -1 and b"b_row_index" in msg
    assert call(a_num_rows=-1)[0] == -1
    assert call(b_num_rows=-1)[0] == -1
    assert call(c_num_rows=-1)[0] == -1
    rc, msg = call(c=12288 + 1)
    assert rc == -2 and b"element size" in msg


def test_workspace_bytes_for_needs_no_device():
    """gg_workspace_bytes_for: nothing for calls that can never cut tiles along the depth, the
    full workspace for deep products and weight gradients."""
    lib = ctypes.CDLL(HIP_LIB)
    lib.gg_workspace_bytes_for.argtypes = [ctypes.c_void_p]
    lib.gg_workspace_bytes_for.restype = ctypes.c_uint64
    full = 4096 + 256 * 256 * 256 * 4

    def want(**kw):
        g = _Args()
        g.struct_bytes = ctypes.sizeof(_Args)
        g.a, g.b, g.c = 4096, 8192, 12288
        g.num_groups, g.tokens, g.hidden_in, g.hidden_out = 8, 32768, 4096, 14336
        for k, v in kw.items():
            setattr(g, k, v)
        return lib.gg_workspace_bytes_for(ctypes.byref(g))

    assert lib.gg_workspace_bytes_for(None) == 0
    assert want(struct_bytes=4) == 0
    assert want() == 0                                     # 64 depth slices: too shallow
    assert want(hidden_in=14336, hidden_out=4096) == full  # 224 slices
    assert want(hidden_in=6144) == full and want(hidden_in=6080) == 0
    # the depth is a group's rows, and one group may hold them all (deep groups among shallow ones
    # are cut along the depth)
    assert want(trans_a=1) == full
    assert want(trans_a=1, tokens=6144) == full and want(trans_a=1, tokens=6080) == 0
    assert want(trans_a=1, tokens=65536, hidden_in=4097) == 0   # general kernels
    assert want(trans_a=1, tokens=65536, a=4096 + 2) == 0       # off the 4-byte boundary
    assert want(hidden_in=14336, a_row_index=64) == 0      # scattered or gathered tiles stay whole
    assert want(hidden_in=14336, hidden_out=2048, epilogue=1) == 0
    assert want(hidden_in=14336, flags=1) == 0 and want(hidden_in=14336, flags=4) == 0
    assert want(dtype=2, hidden_in=12288) == full and want(dtype=2, hidden_in=12160) == 0
    # even sizes that are no multiples of 8: only where the caller says so
    for sizes in (dict(hidden_in=14334), dict(hidden_in=14336, hidden_out=4094), dict(trans_a=1, hidden_out=4098)):
        assert want(**sizes) == 0 and want(flags=128, **sizes) == 0 and want(flags=256, **sizes) == full
        assert want(flags=256 | 1, **sizes) == 0 and want(flags=256, c_row_index=64 * (sizes.get("trans_a") is None), **sizes) == (
            full if "trans_a" in sizes else 0)


def test_workspace_bytes_for_strided_operands():
    """gg_workspace_bytes_for_strided: by the call's own sizes, whatever they are (gg_workspace_bytes_for has nothing for
    odd hidden sizes: its calls run those on the general kernels)."""
    lib = ctypes.CDLL(HIP_LIB)
    for f in (lib.gg_workspace_bytes_for_strided, lib.gg_workspace_bytes_for):
        f.restype = ctypes.c_uint64
    lib.gg_workspace_bytes_for_strided.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_int64]
    lib.gg_workspace_bytes_for.argtypes = [ctypes.c_void_p]
    full = 4096 + 256 * 256 * 256 * 4

    def want(a_row, b_row, plain, **kw):
        g = _Args()
        g.struct_bytes = ctypes.sizeof(_Args)
        g.a, g.b, g.c = 4096, 8192, 12288 + 2
        g.num_groups, g.tokens, g.hidden_in, g.hidden_out = 8, 32768, 14335, 4095
        for k, v in kw.items():
            setattr(g, k, v)
        assert lib.gg_workspace_bytes_for(ctypes.byref(g)) == plain
        return lib.gg_workspace_bytes_for_strided(ctypes.byref(g), a_row, b_row)

    assert lib.gg_workspace_bytes_for_strided(None, 8, 8) == 0
    assert want(14336, 4096, 0) == full and want(14336, 14336, 0, trans_b=1) == full
    assert want(14336, 4096, 0, trans_a=1) == full
    assert want(6144, 4096, 0, hidden_in=6143) == full and want(6080, 4096, 0, hidden_in=6079) == 0
    # groups of few rows: as for the same call on whole chunks
    few = dict(num_groups=16, tokens=960, hidden_out=2047, dtype=1)
    assert want(6144, 2048, 0, hidden_in=6144, **few) == want(6144, 2048, full, **{**few, "hidden_in": 6144, "hidden_out": 2048, "c": 12288})
    assert want(14336, 4096, 0, struct_bytes=4) == 0 and want(14336, 4096, 0, flags=1) == 0
    # (strides that gg_gmm_strided refuses, and what it does not take)
    assert want(14328, 4096, 0) == 0 and want(14336, 4100, 0) == 0 and want(14336, 4096, 0, a=4096 + 8) == 0
    assert want(14336, 4096, 0, dtype=2) == 0 and want(14336, 4096, 0, epilogue=1) == 0 and want(1 << 22, 4096, 0) == 0


def test_tile_shapes_need_no_device():
    """The tile shape each call of the GPU tests of tile shapes runs on, so that a moved threshold cannot leave a
    shape without a test; and the general kernels, where a half of gate | up is no multiple of 8."""
    from test_gmm_gpu import _TILE_SHAPES, _TILE_SHAPES_F8
    lib = ctypes.CDLL(HIP_LIB)
    lib.gg_debug_tile.argtypes = [ctypes.c_void_p] * 3
    lib.gg_workspace_bytes_for.argtypes = [ctypes.c_void_p]
    lib.gg_workspace_bytes_for.restype = ctypes.c_uint64

    def call(sizes, hin, hout, **kw):
        g, bm, bn = _Args(), ctypes.c_int(-1), ctypes.c_int(-1)
        g.struct_bytes = ctypes.sizeof(_Args)
        g.a, g.b, g.c = 4096, 8192, 12288
        g.num_groups, g.tokens, g.hidden_in, g.hidden_out = len(sizes), sum(sizes), hin, hout
        for k, v in kw.items():
            setattr(g, k, v)
        assert lib.gg_debug_tile(ctypes.byref(g), ctypes.byref(bm), ctypes.byref(bn)) == 0
        return (bm.value, bn.value), lib.gg_workspace_bytes_for(ctypes.byref(g)) > 0

    for sizes, hin, hout, bm, bn, partial_tiles in _TILE_SHAPES.values():
        scattered_cut = partial_tiles > 0 and bm < 256
        for dtype in (0, 1):
            for trans_b in (0, 1):
                kw = dict(dtype=dtype, trans_b=trans_b)
                assert call(sizes, hin, hout, **kw) == ((bm, bn), partial_tiles > 0)
                assert call(sizes, hin, hout, a_row_index=64, **kw) == ((bm, bn), scattered_cut)
                assert call(sizes, hin, hout // 2, epilogue=1, **kw) == ((bm, bn // 2), scattered_cut)
                assert call(sizes, hin, hout // 2, epilogue=1, a_row_index=64, c_row_index=64, **kw) == ((bm, bn // 2), scattered_cut)
    for sizes, hin, hout, bm, bn, partial_tiles in _TILE_SHAPES_F8.values():
        for dtype in (2, 3):
            assert call(sizes, hin, hout, dtype=dtype, trans_b=1) == ((bm, bn), partial_tiles > 0)
            assert call(sizes, hin, hout, dtype=dtype)[0] == (256, 256)
    assert call([300, 200], 264, 196, epilogue=1) == ((0, 0), False)
    # weight gradients: small tiles up to two rounds of them, where groups are not deep
    assert call([129] * 40, 264, 136, trans_a=1)[0] == (128, 128)
    assert call([64] * 256, 256, 768, trans_a=1)[0] == (256, 256)
    assert call([3000] * 4, 256, 256, trans_a=1)[0] == (256, 256)
    assert lib.gg_debug_tile(None, None, None) == -1


def test_row_index_bounds_reach_every_kernel():
    """The C ABI hands the row counts that bound a row index to the general kernels as it does to
    the streaming ones (checked in the sources: no GPU test feeds bad indices on purpose)."""
    api = open(os.path.join(ROOT, "grouped_gemm_amd", "csrc", "gmm_api.hip")).read()
    for field in ("gp.a_num_rows = index_rows.a", "gp.b_num_rows = index_rows.b", "gp.c_num_rows = index_rows.c",
                  "p.a_index_rows =", "p.c_index_rows ="):
        assert field in api, field
    generic = open(os.path.join(ROOT, "grouped_gemm_amd", "csrc", "gmm_generic.hpp")).read()
    assert "strided < index_rows" in generic and "mem_row >= gp.c_num_rows" in generic


def test_padded_sizes_stay_below_the_limit_of_hidden_sizes():
    # A size that whole 16-byte chunks bring to a legal size (below 2 ** 22) is padded to a legal one.
    from grouped_gemm_amd.backend import _padded_size
    limit = 1 << 22
    for itemsize in (1, 2):
        chunk = 16 // itemsize
        for n in (*range(1, 3000, 7), *range(limit - 300, limit)):
            padded, least = _padded_size(n, itemsize), (n + chunk - 1) // chunk * chunk
            assert padded >= least and padded % chunk == 0
            assert padded < limit or least == limit, (n, itemsize)
            assert padded - n <= max(chunk, n // 8), (n, itemsize)


def _pair(lib, sizes, hin, hout, trans_b, dtype=0, workspaces=((0, 0), (0, 0)), strides=None, **kw):
    """(status, tile shapes) of the two gradients of a product hin -> hout in one call, sizes on the host; addresses are
    never dereferenced."""
    rows = (ctypes.c_int64 * len(sizes))(*sizes)
    both = []
    for weight, (at, length) in zip((False, True), workspaces):
        g = _Args()
        g.struct_bytes, g.dtype = ctypes.sizeof(_Args), dtype
        g.a, g.b, g.c = 4096, 8192, 12288
        g.batch_sizes, g.num_groups, g.tokens = ctypes.addressof(rows), len(sizes), sum(sizes)
        g.trans_a, g.trans_b = int(weight), int(not weight and not trans_b)
        g.hidden_in, g.hidden_out = (hin, hout) if weight and not trans_b else (hout, hin)
        g.workspace, g.workspace_bytes, g.flags = at, length, 128
        for k, v in kw.items():
            setattr(g, k, v)
        both.append(g)
    shapes = (ctypes.c_int * 4)(*[-1] * 4)
    status = lib.gg_debug_pair(ctypes.byref(both[0]), ctypes.byref(both[1]), strides and (ctypes.c_int64 * 4)(*strides), shapes)
    return status, tuple(shapes)


def test_pairs_that_share_a_workspace():
    """Two calls in one launch need workspaces that do not overlap: the same one twice means two launches; parts of one
    are refused, as one call's partial tiles would land on the other's arrival counters."""
    lib = ctypes.CDLL(HIP_LIB)
    lib.gg_last_error.restype = ctypes.c_char_p
    least, at = 4096 + 256 * 256 * 4, 1 << 32
    deep = ([700, 0, 5300], 264, 8192, False)   # pieces in both: 128 slices, and up to 94
    assert _pair(lib, *deep, workspaces=((at, least), (at + least, least))) == (0, (128, 256, 128, 128))
    assert _pair(lib, *deep, workspaces=((at, least), (at, least))) == (0, (0, 0, 0, 0))
    for shift in (256, 4096, least - 256):
        for first, second in ((at, at + shift), (at + shift, at)):
            assert _pair(lib, *deep, workspaces=((first, least), (second, least)))[0] == -1
            assert b"overlap" in lib.gg_last_error()
    # nothing is cut in either: neither touches a workspace
    assert _pair(lib, [60, 50], 64, 72, True, workspaces=((at, least), (at + 256, least))) == (0, (64, 128, 128, 128))


def test_pairs_by_weights_and_rounds():
    """Which gradients take one launch: few rows to a group up to 384 MB of weights, others below eight rounds of tiles of
    either product."""
    lib = ctypes.CDLL(HIP_LIB)
    one = lambda *args, **kw: any(_pair(lib, *args, **kw)[1])
    assert one([19] * 38, 1944, 2496, False) and one([65] * 45, 1064, 1184, True)
    assert one([6] * 96, 1024, 2048, False) and not one([6] * 97, 1024, 2048, False)          # 384 MB and 388
    assert not one([9] * 13, 3856, 4744, True) and not one([23] * 108, 3792, 9328, False)
    assert one([1024] * 16, 2048, 4096, False) and not one([4096] * 8, 4096, 14336, False)   # 4 rounds of one, 8 of both
    assert one([4096] * 8, 4096, 1408, False)                                                 # 8 and 3
    assert not one([600] * 513, 64, 64, False)                                                # more groups than one launch takes


def test_every_pair_kernel_has_a_case():
    """The tiles that each case of the GPU test of pair kernels takes, so that a moved threshold cannot leave a kernel
    without a test: every one of the library's pairs, of both element types, on multiples of 8 and on odd sizes."""
    import re
    from test_gmm_gpu import _PAIR_SHAPES, _row_stride
    lib = ctypes.CDLL(HIP_LIB)
    names = {(256, 256): "Wide", (128, 256): "Short", (64, 128): "Small", (128, 128): "SmallSquare"}
    reached = {False: set(), True: set()}
    for experts, rows, hin, hout, trans_b, first, second in _PAIR_SHAPES:
        odd = hin % 8 != 0 or hout % 8 != 0
        sizes = [rows // experts] * (experts - 1) + [rows - rows // experts * (experts - 1)]
        in_row, out_row = _row_stride(hin), _row_stride(hout)
        strides = (out_row, in_row if trans_b else out_row, *((out_row, in_row) if trans_b else (in_row, out_row))) if odd else None
        for dtype in (0, 1):
            assert _pair(lib, sizes, hin, hout, trans_b, dtype=dtype, strides=strides) == (0, first + second)
            reached[odd].add(("kBF16 kF16".split()[dtype], "kNN" if trans_b else "kNT", names[first], names[second]))
    built = open(os.path.join(ROOT, "grouped_gemm_amd", "csrc", "gmm_variants.def")).read()
    pairs = set(re.findall(r"^GG_PAIR\(\d+, (\w+), (\w+), (\w+), (\w+)\)", built, flags=re.M))
    assert len(pairs) == 24 and reached[False] == pairs and reached[True] == pairs


def test_entry_points_beside_gg_gmm_refuse_bad_arguments():
    """gg_gmm_pair, gg_gmm_strided, gg_gmm_pair_strided, gg_keeps_gate_up and gg_gmm_keep_gate_up: every case fails before the
    device is looked for."""
    lib = ctypes.CDLL(HIP_LIB)
    lib.gg_last_error.restype = ctypes.c_char_p
    rows = (ctypes.c_int64 * 2)(3, 5)
    i64 = ctypes.c_int64

    def args(**kw):
        g = _Args()
        g.struct_bytes = ctypes.sizeof(_Args)
        g.a, g.b, g.c = 4096, 8192, 12288
        g.batch_sizes, g.num_groups, g.tokens, g.hidden_in, g.hidden_out = ctypes.addressof(rows), 2, 8, 136, 264
        for k, v in kw.items():
            setattr(g, k, v)
        return ctypes.byref(g)

    for bad in (None, args(struct_bytes=8)):
        assert lib.gg_gmm_pair(bad, args()) == -1 and lib.gg_gmm_pair(args(tokens=0), bad) == -1
        assert lib.gg_gmm_pair_strided(bad, i64(136), i64(264), args(), i64(136), i64(264)) == -1
        assert lib.gg_gmm_strided(bad, i64(136), i64(264)) == -1
        assert lib.gg_debug_pair(bad, args(), None, (ctypes.c_int * 4)()) == -1
        assert lib.gg_keeps_gate_up(bad) == 0 and lib.gg_gmm_keep_gate_up(bad, ctypes.c_void_p(4096)) == -1
    assert lib.gg_debug_pair(args(), args(), None, None) == -1
    assert lib.gg_gmm_pair(args(trans_a=1, trans_b=1), args(trans_a=1)) == -1      # the first call alone is wrong,
    assert lib.gg_gmm_pair(args(tokens=0), args(trans_a=1, tokens=7)) == -1       # the second alone (sizes past its rows)
    for a_row, b_row, kw in ((132, 264, {}), (128, 264, {}), (136, 256, {}), (136, 264 + 4, {}), (1 << 22, 264, {}),
                             (136, 264, dict(a=4096 + 8)), (136, 264, dict(b=8192 + 2)), (136, 264, dict(dtype=2)),
                             (136, 264, dict(epilogue=1)), (136, 264, dict(trans_a=1, accumulate_f32=1)),
                             (136, 264, dict(a_row_index=64)), (136, 128, dict(trans_b=1)), (264, 136, dict(trans_a=1))):
        assert lib.gg_gmm_strided(args(**kw), i64(a_row), i64(b_row)) == -1, (a_row, b_row, kw)
        assert b"strides" in lib.gg_last_error()
        assert lib.gg_gmm_pair_strided(args(**kw), i64(a_row), i64(b_row), args(), i64(136), i64(264)) == -1
    swiglu = dict(epilogue=1)
    assert lib.gg_keeps_gate_up(args(**swiglu)) == 1 and lib.gg_keeps_gate_up(args(dtype=1, **swiglu)) == 1
    for kw in (dict(epilogue=0), dict(dtype=2, **swiglu), dict(hidden_in=132, **swiglu), dict(hidden_out=260, **swiglu),
               dict(c=12288 + 8, **swiglu), dict(c_row_index=64, **swiglu)):
        assert lib.gg_keeps_gate_up(args(**kw)) == 0 and lib.gg_gmm_keep_gate_up(args(**kw), ctypes.c_void_p(4096)) == -1
    for at in (0, 4096 + 8, 4096 + 2):
        assert lib.gg_gmm_keep_gate_up(args(**swiglu), ctypes.c_void_p(at)) == -1
        assert b"16-byte" in lib.gg_last_error()


def _deep_cut(lib, rows, per_group, workgroups, partial_tiles, tile_outputs):
    sizes, pieces, tiles = (ctypes.c_int64 * len(rows))(*rows), ctypes.c_int(-1), ctypes.c_int(-1)
    assert lib.gg_debug_deep_cut(sizes, ctypes.c_int64(len(rows)), ctypes.c_int64(per_group), workgroups, partial_tiles,
                                 tile_outputs, ctypes.byref(pieces), ctypes.byref(tiles)) == 0
    return pieces.value, tiles.value


def test_deep_tiles_are_cut_to_end_the_launch_soonest():
    """Into how many pieces a weight gradient cuts its deepest tiles, against all tiles laid out one by one."""
    lib = ctypes.CDLL(HIP_LIB)
    small = 128 * 128
    # one deep group of more tiles than there are workgroups for four pieces each, in front of shallow ones: two pieces of all
    # 84 tiles (71 slices), not four of 64 (20 whole tiles of 141 slices)
    assert _deep_cut(lib, [9000, 30, 0, 1400], 84, 256, 1024, small) == (2, 84)
    assert _deep_cut(lib, [9000], 84, 256, 1024, small) == (2, 84)
    assert _deep_cut(lib, [9000, 30, 0, 1400], 64, 256, 1024, small) == (4, 64)
    assert _deep_cut(lib, [9000, 8900], 32, 256, 1024, small) == (4, 64)
    assert _deep_cut(lib, [13000, 50, 12800], 32, 256, 256, 256 * 256) == (4, 64)
    assert _deep_cut(lib, [3000] * 4, 64, 256, 1024, small) == (0, 0)      # a round of equal tiles
    assert _deep_cut(lib, [9000, 30], 84, 256, 0, small) == (0, 0)         # nowhere to put partial tiles
    assert _deep_cut(lib, [0, 0], 4, 256, 1024, small) == (0, 0)

    rng = np.random.default_rng(11)
    for _ in range(400):
        groups = int(rng.integers(1, 40))
        rows = (rng.pareto(1.0, groups) * 600).clip(0, 60000).astype(int).tolist()
        per_group, workgroups, slots = int(rng.integers(1, 120)), int(rng.choice([256, 512])), int(rng.choice([0, 100, 256, 1024]))
        tile_outputs = int(rng.choice([small, 256 * 256]))
        least = 16 if tile_outputs == small else 48
        depths = [-(-r // 64) for r in sorted(rows, reverse=True) for _ in range(per_group)]
        share = (sum(rows) + groups * 32) // 64 * per_group // workgroups
        chosen, best = (0, 0), depths[0]
        for n in (4, 2):
            deep_enough = sum(2 * d > share and d >= n * least for d in depths)
            cut = min(deep_enough, workgroups // n, slots // n, 1024)
            length = max(-(-depths[0] // n), depths[cut] if cut < len(depths) else 0)
            if cut > 0 and length < best:
                chosen, best = (n, cut), length
        assert _deep_cut(lib, rows, per_group, workgroups, slots, tile_outputs) == (chosen if depths[0] > share else (0, 0))
    assert lib.gg_debug_deep_cut(None, ctypes.c_int64(1), ctypes.c_int64(1), 256, 0, small, None, None) == -1


def _pieces(lib, rows, per_group, workgroups, units, partial_tiles, tile_outputs, tail=1):
    sizes, pieces = (ctypes.c_int64 * len(rows))(*rows), (ctypes.c_int32 * len(rows))()
    places = (ctypes.c_int32 * (4 * workgroups))()
    assert lib.gg_debug_pieces(sizes, ctypes.c_int64(len(rows)), ctypes.c_int64(per_group), workgroups, units, partial_tiles,
                               tile_outputs, tail, pieces, places, ctypes.c_int64(workgroups)) == 0
    return list(pieces), np.array(places[:4 * per_group * sum(pieces)]).reshape(-1, 4)


def test_pieces_of_one_length():
    """How a weight gradient is cut into pieces of one length: every piece once, in its own place, within what there is."""
    lib = ctypes.CDLL(HIP_LIB)
    small, full = 128 * 128, 256 * 256
    # pieces per tile, deepest group first (in brackets us of the launch, and of others)
    assert _pieces(lib, [8483] * 4, 11, 512, 256, 1024, small, 8)[0] == [5] * 4              # (29.8; 4: 30.3, 3: 34.5)
    assert _pieces(lib, [20000] * 2, 22, 512, 256, 1024, small, 8)[0] == [5] * 2             # (44.5; 4: 49, 6: 48.3)
    assert _pieces(lib, [6377] * 7, 12, 512, 256, 1024, small, 4)[0] == [3] * 7              # (31.0; 2: 36.5, 4: 36.0)
    assert _pieces(lib, [17150, 7470, 4590, 3250, 2490, 2000, 1660, 1390], 8, 512, 256, 1024, small)[0] == [12, 6, 4, 3, 2, 0, 0, 0]
    assert _pieces(lib, [6000] * 6, 8, 512, 256, 1024, small, 4)[0] == [0] * 6              # the last round's cut is as good (25.7; 5: 26.7)
    assert _pieces(lib, [4000] * 4, 16, 512, 256, 1024, small, 4)[0] == [0] * 4
    assert _pieces(lib, [4215, 1834, 1129, 799, 611, 491, 408, 347, 302, 266], 132, 512, 256, 1024, small)[0][:2] == [2, 0]   # whole ones share too
    zipf = [5696, 2432, 1600, 1088, 832, 704, 640, 512] + [300] * 48
    assert _pieces(lib, zipf, 18, 256, 256, 256, full)[0][:3] == [4, 2, 0]                   # (91.5; 5 and 3: 93.5)
    assert _pieces(lib, [3000] * 4, 64, 512, 256, 0, small)[0] == [0] * 4                    # nowhere to put partial tiles
    assert _pieces(lib, [1500, 20], 4, 512, 256, 1024, small)[0][0] > 1 and _pieces(lib, [1500], 4, 256, 256, 1024, full)[0] == [0]
    assert _pieces(lib, [0, 0], 4, 512, 256, 1024, small)[0] == [0, 0]
    rng = np.random.default_rng(5)
    seen = dict(all_cut=0, some_cut=0, none=0, few_slots=0)
    for trial in range(600):
        groups = int(rng.integers(1, 513 if trial % 4 == 0 else 40))
        rows = (rng.pareto(0.7, groups) * rng.choice([60, 600, 4000])).clip(0, 2**31 // groups - 1).astype(int).tolist()
        if trial % 3 == 0:
            rows = rng.integers(4000, 12000, groups := int(rng.integers(1, 12))).tolist()
        tile_outputs = int(rng.choice([small, full]))
        units = 256
        workgroups = units * (2 if tile_outputs == small else 1)
        per_group, slots = int(rng.choice([1, 4, 11, 30, 120])), int(rng.choice([1, 20, 100, 256, 1024]))
        pieces, places = _pieces(lib, rows, per_group, workgroups, units, slots, tile_outputs, int(rng.choice([1, 1, 2, 4])))
        depths = [-(-r // 64) for r in sorted(rows, reverse=True)]
        cut = sum(n > 0 for n in pieces)
        assert all(n > 0 for n in pieces[:cut])                    # the deepest groups
        assert cut * per_group <= 1024                            # one arrival counter per tile
        assert len(places) <= min(workgroups, slots)              # at most one piece to a workgroup, a place for each
        assert all(2 <= n <= 17 for n in pieces[:cut])
        if cut:
            length = max(-(-d // n) for d, n in zip(depths, pieces[:cut]))
            assert length >= (6 if tile_outputs == small else 16)
            assert all(d > 1.5 * (length - 1) for d in depths[:cut]) and all(d < 2 * length + 2 for d in depths[cut:])
            tile, piece, of, slot = places.T
            assert len({(t, p) for t, p in zip(tile, piece)}) == len(places) and sorted(slot) == list(range(len(places)))
            assert (of == np.array(pieces)[tile // per_group]).all() and (piece < of).all() and tile.max() < cut * per_group
        seen["all_cut"] += cut == groups
        seen["none"] += cut == 0
        seen["some_cut"] += 0 < cut < groups
        seen["few_slots"] += cut > 0 and len(places) > slots // 2
    assert all(n >= 40 for n in seen.values()), seen
    bad = (ctypes.c_int32 * 4)()
    assert lib.gg_debug_pieces(None, ctypes.c_int64(1), ctypes.c_int64(1), 512, 256, 1, small, 1, bad, None, ctypes.c_int64(0)) == -1
    one = (ctypes.c_int64 * 1)(9000)
    assert lib.gg_debug_pieces(one, ctypes.c_int64(1), ctypes.c_int64(4), 512, 256, 1024, small, 1, bad, (ctypes.c_int32 * 4)(), ctypes.c_int64(1)) == -1


# ----------------------------------------------------------------- workloads

def test_workload_generators():
    from grouped_gemm_amd import workloads
    g = torch.Generator().manual_seed(0)
    s2 = workloads.router_sizes(16384, 8, 2, g)
    assert int(s2.sum()) == 32768 and s2.numel() == 8 and int(s2.min()) > 0
    s3 = workloads.zipf_sizes(49152, 64, 1.2, 4, g)
    assert int(s3.sum()) == 49152 and int((s3 == 0).sum()) >= 4
    s5 = workloads.poisson_sizes(65536, 256, g)
    assert int(s5.sum()) == 65536 and s5.numel() == 256 and int(s5.min()) >= 0
    w = workloads.make(3, device="cpu", shrink=16)
    assert w.a.shape == (49152 // 16, 128) and w.b.shape == (64, 128, 88) and not w.trans_b
    assert int(w.batch_sizes.sum()) == w.tokens
    w5 = workloads.make(5, device="cpu", shrink=32)
    assert w5.trans_b and w5.b.shape == (256, 64, 224)
    assert w5.flops_per_gemm() == 2 * w5.tokens * 224 * 64


# -------------------------------------------------------------- golden fixture

def test_config1_fixture_matches_oracle(oracle):
    spec = importlib.util.spec_from_file_location(
        "make_config1", os.path.join(ROOT, "tests", "golden", "make_config1.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    a, b, grad, sizes = mod.inputs()
    fwd, agrad, bgrad = mod.expected(a, b, grad, sizes)
    gold = np.load(os.path.join(ROOT, "tests", "golden", "config1.npz"))
    assert np.array_equal(gold["fwd"], fwd[::8].numpy())
    assert np.array_equal(gold["agrad"], agrad[::8].numpy())
    assert np.array_equal(gold["bgrad"], bgrad[:, ::8].numpy())
    # the same numbers from the library routine, by autograd through the loop
    out, ag, bg = oracle.gmm_autograd_loop(a, b, sizes, False, grad)
    torch.testing.assert_close(out, fwd, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(ag, agrad, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(bg, bgrad, rtol=1e-5, atol=1e-4)


# ----------------------------------------------------------------- traceable operator

def test_traceable_gradients_shapes_without_a_device():
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    from grouped_gemm_amd import ops  # noqa: F401 (registers the operators)
    for trans_b, shape in ((False, (4, 64, 96)), (True, (4, 96, 64))):
        with FakeTensorMode():
            a, b = torch.empty(100, 64, dtype=torch.bfloat16), torch.empty(shape, dtype=torch.bfloat16)
            grad, sizes = torch.empty(100, 96, dtype=torch.bfloat16), torch.empty(4, dtype=torch.int64)
            agrad, bgrad = torch.ops.grouped_gemm_amd.gmm_gradients(grad, a, b, sizes, trans_b)
        assert agrad.shape == (100, 64) and bgrad.shape == shape


def test_traceable_operator_shapes_without_a_device():
    # the torch.library form of the operator: output shapes for all three layouts from fake
    # tensors alone (what torch.compile needs), no kernel runs
    from torch._subclasses.fake_tensor import FakeTensorMode
    from grouped_gemm_amd import ops
    with FakeTensorMode():
        a = torch.empty(100, 64, dtype=torch.bfloat16)
        bs = torch.empty(4, dtype=torch.int64)
        assert ops.gmm_traceable(a, torch.empty(4, 64, 96, dtype=torch.bfloat16), bs).shape == (100, 96)
        assert ops.gmm_traceable(a, torch.empty(4, 96, 64, dtype=torch.bfloat16), bs, trans_b=True).shape == (100, 96)
        wgrad = torch.ops.grouped_gemm_amd.gmm(a, torch.empty(100, 96, dtype=torch.bfloat16), bs, True, False)
        assert wgrad.shape == (4, 64, 96) and wgrad.dtype == torch.bfloat16



def _early_loads(lines):
    """Loads straight to LDS in a disassembly (branch targets as labels) that are not what they were written as, on any way that leads to
    them: less than five wait states behind a vector instruction that writes a word of their descriptor (the hardware does not wait for it,
    and the compiler does not look into the assembly that these loads are written in), right behind the write of m0 that aims
    them, aimed by another instruction than theirs, or by one that has aimed a load already."""
    functions, code, labels = [], [], {}
    for line in lines:
        m = re.match(r"\s+([a-z]\w+)\s*(.*?)\s*(//.*)?$", line)
        if m:
            code.append((m.group(1), m.group(2)))
        elif m := re.match(r"(?:[0-9a-f]+ )?<(L\d+)>:", line):
            labels[m.group(1)] = len(code)
        elif re.match(r"[0-9a-f]+ <", line):
            functions.append((code, labels))
            code, labels = [], {}
    functions.append((code, labels))
    bad, loads = [], 0
    for code, labels in functions:
        jumps = {}
        for i, (op, args) in enumerate(code):
            if op == "s_branch" or op.startswith("s_cbranch"):
                jumps.setdefault(labels[args.split()[0]], []).append(i)

        def ways_to(i):
            falls = i > 0 and code[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64")
            return jumps.get(i, []) + ([i - 1] if falls else [])

        def to_lds(op, args):
            return op == "buffer_load_dwordx4" and args.endswith(" lds")

        def wrong(i):
            first, last = map(int, re.search(r", s\[(\d+):(\d+)\]", code[i][1]).groups())
            todo, least = [(k, 0, False) for k in ways_to(i)], {}
            if not todo:
                return True
            while todo:
                k, waited, aimed = todo.pop()
                if least.get((k, aimed), 9) <= waited:
                    continue
                least[k, aimed] = waited
                op, args = code[k]
                m = re.match(r"s(?:(\d+)|\[(\d+):(\d+)\])", args) if op.startswith("v_") else None
                if m and waited < 5 and int(m.group(1) or m.group(2)) <= last and int(m.group(1) or m.group(3)) >= first:
                    return True
                if not aimed and re.match(r"m0\b", args):
                    if op != "s_add_u32" or waited == 0:
                        return True
                    aimed = True
                elif not aimed and to_lds(op, args):
                    return True
                waited = min(waited + (1 + int(args, 0) if op == "s_nop" else 1), 5)
                if waited < 5 or not aimed:
                    ways = ways_to(k)
                    if not ways and not aimed:
                        return True
                    todo += [(way, waited, aimed) for way in ways]
            return False

        for i, (op, args) in enumerate(code):
            if to_lds(op, args):
                loads += 1
                if wrong(i):
                    bad.append(code[max(i - 8, 0):i + 1])
    return bad, loads


def _code_objects(folder):
    """llvm-objdump and the device code of the built library, one file per translation unit."""
    objdump = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
    if not os.path.exists(objdump):
        pytest.skip("no llvm-objdump")
    copy = folder / "library.so"
    copy.write_bytes(open(os.path.join(ROOT, "grouped_gemm_amd", "libgrouped_gemm_hip.so"), "rb").read())
    subprocess.run([objdump, "--offloading", str(copy)], check=True, capture_output=True)
    objects = [f for f in sorted(folder.iterdir()) if "gfx950" in f.name]
    assert objects
    return objdump, objects


def test_loads_to_lds_are_late_enough(tmp_path):
    # the check itself ...
    load = "\tbuffer_load_dwordx4 v1, s[8:11], 0 offen lds"
    aim = "\ts_add_u32 m0, s3, 16"
    word = "\tv_readfirstlane_b32 s9, v0"
    for code, bad in [
            ([word, aim, "\ts_nop 0", load], 1), ([word, aim, "\ts_nop 2", load], 1), ([word, aim, "\ts_nop 3", load], 0),
            (["\tv_readfirstlane_b32 s12, v0", aim, "\ts_nop 0", load], 0), (["\tv_cmp_eq_u32_e64 s[10:11], v0, v1", aim, "\ts_nop 0", load], 1),
            (["\ts_nop 4", aim, load], 1),                                             # right behind its aim
            ([aim, "\ts_mov_b32 m0, s4", "\ts_nop 4", load], 1),                        # aimed elsewhere
            (["\ts_nop 4", load], 1), ([aim, "\ts_nop 0", load, "\ts_nop 0", load], 1),   # not aimed, aimed once for two
            # the word is written at the end of a loop, far from its beginning in the text, and jumped over in between
            ([aim, "<L0>:", "\ts_nop 0", load, "\ts_nop 7", aim, word, "\ts_cbranch_scc1 L0"], 1),
            ([aim, "<L0>:", "\ts_nop 3", load, "\ts_nop 7", aim, word, "\ts_cbranch_scc1 L0"], 0),
            ([aim, "<L0>:", "\ts_nop 3", load, "\ts_nop 7", "\ts_cbranch_scc1 L0"], 1),   # (aimed for the first time round only)
            ([word, "\ts_branch L1", "\ts_nop 7", "<L1>:", aim, "\ts_nop 0", load], 1),
            (["\ts_cbranch_scc0 L1", word, "\ts_nop 4", "\ts_branch L2", "<L1>:", "\ts_nop 0", "<L2>:", aim, "\ts_nop 0", load], 0)]:
        early, loads = _early_loads(code)
        assert (len(early), loads) == (bad, sum(line == load for line in code)), code
    # ... and every kernel that was built
    objdump, objects = _code_objects(tmp_path)
    total = 0
    for f in objects:
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--symbolize-operands", str(f)], check=True, capture_output=True, text=True).stdout
        early, loads = _early_loads(text.splitlines())
        assert not early, (f.name, early[:3])
        total += loads
    assert total > 1000


def test_first_slice_of_weight_gradients_moves_few_sums(tmp_path):
    """Weight gradients on full tiles: sums that the slices move from their accumulation registers to others, and back."""
    objdump, objects = _code_objects(tmp_path)
    moves = {}
    for f in objects:
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True, text=True).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(_ZN2gg10gmm_kernelILi[01]ELi2ELi256ELi256E(?:Li\d+E){4}Li0E\w+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)",
                                     text, flags=re.S | re.M):
            blocks = [re.findall(r"^\s+(\w+)", b, flags=re.M) for b in re.split(r"\bs_c?branch\w*", body)]
            moves[name] = sum(b.count("v_accvgpr_read_b32") for b in blocks if sum("mfma" in op for op in b) >= 32)
    assert len(moves) == 2 and max(moves.values()) <= 12, moves


def test_reading_accumulation_keeps_its_registers(tmp_path):
    """Full tiles that add to fp32 by reading, adding and writing (epilogue 1 of the template's arguments) have no scratch memory: with
    some, each block row of c began with a reload that waited for all stores of the one before."""
    objdump, objects = _code_objects(tmp_path)
    found = {}
    for f in objects:
        notes = subprocess.run([objdump.replace("objdump", "readelf"), "--notes", str(f)], check=True, capture_output=True, text=True).stdout
        for name, scratch in re.findall(r"\.name:\s+(_Z\w+)\n.*?\.private_segment_fixed_size:\s+(\d+)", notes, flags=re.S):
            found[name] = int(scratch)
    reading = {name: n for name, n in found.items() if re.search(r"10gmm_kernelILi\dELi2ELi256E(Li\d+E){5}Li1E", name)}
    assert len(reading) == 4 and not any(reading.values()), reading
