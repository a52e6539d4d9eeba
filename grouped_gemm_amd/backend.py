"""Output allocation and the call into the native extension.

Mirror of the reference's grouped_gemm/backend.py:11-28: same function names, same
argument meaning, same assertions, same uninitialised output.  The extension is
required: there is no fallback path.
"""
# torch must be imported before the extension so that libc10 resolves
# (grouped_gemm/backend.py:1-3).
import torch

try:
    from grouped_gemm_amd import grouped_gemm_backend as backend
except ImportError as exc:  # pragma: no cover - depends on the build
    raise ImportError(
        "grouped_gemm_amd: the native extension grouped_gemm_backend is not built or cannot be "
        "loaded (" + str(exc) + "). Build it with `python grouped_gemm_amd/build.py`; it needs "
        "hipcc, ROCm and PyTorch-ROCm. There is no fallback implementation."
    ) from exc

# The reference installs its extension under the top-level name grouped_gemm_backend
# (setup.py:35, imported at grouped_gemm/backend.py:8); keep that name importable.
import sys as _sys
_sys.modules.setdefault("grouped_gemm_backend", backend)


def _check_ranks(a, b, batch_sizes, trans_a, trans_b):
    assert not (trans_a and trans_b)
    assert batch_sizes.ndim == 1, "Expected 1d tensor for batch_sizes"
    assert a.ndim == 2, "Expected 2d tensor for 'a'"
    assert b.ndim == (2 if trans_a else 3)


def _allocate_output(a, b, batch_sizes, trans_a, trans_b):
    _check_ranks(a, b, batch_sizes, trans_a, trans_b)
    shape = (
        (batch_sizes.shape[0], a.shape[1], b.shape[1])
        if trans_a else
        (a.shape[0], (b.shape[1] if trans_b else b.shape[2]))
    )
    return torch.empty(*shape, device=a.device, dtype=_output_dtype(a.dtype))


def _output_dtype(dtype):
    # float8 operands (an addition to the reference, which takes bfloat16 only) give a bfloat16 output
    return torch.bfloat16 if dtype in (torch.float8_e4m3fn, torch.float8_e5m2) else dtype


# Hidden sizes that are not multiples of 8 elements (16 for float8), and operands that do not
# start on a 16-byte boundary, would run on the extension's general kernels, which are many times
# slower than the streaming ones (calling the extension directly gets exactly that, copy-free).
# gmm instead copies operands whose rows cannot be read as they are into tensors with zero-padded, aligned
# rows and runs the streaming kernels on those: one pass over each, still several times faster.  Zeros along
# the depth add nothing to any sum.  Results of two-byte types are written where they belong, whatever their
# rows are; for float8, whose kernels need whole chunks, all three are padded and the result is copied back.
# Needing no copies: two-byte operands on 4-byte boundaries whose hidden sizes are both even.


def _padded_size(n, itemsize):
    """The hidden size that n is padded to: what the streaming kernels need (16-byte rows), and where that adds
    little, rows of whole lines (128 bytes), or sectors (64), which neither loads nor stores share with the
    next row.  8 x 1024 rows, 2047 -> 5461, forward and gradients, padded to 5464 / 5504: 910 / 869 us
    (with results padded too).  Where that would reach the limit of hidden sizes, 2 ** 22, whole chunks again."""
    align = 128 if n * itemsize >= 2048 else (64 if n * itemsize >= 512 else 16)
    for m in (align // itemsize, 16 // itemsize):
        padded = (n + m - 1) // m * m
        if padded < 1 << 22:
            break
    return padded


def _needs_padding(a, b, c, batch_sizes, trans_a, trans_b):
    """Whether gmm goes through zero-padded copies; False when the operands are not the well-formed
    GPU tensors that way assumes (the plain call then runs and raises what it has to raise).  `c`:
    the output, or None for one still to be allocated."""
    if not (a.is_cuda and b.is_cuda and a.dtype == b.dtype and a.dim() == 2 and
            b.dim() == (2 if trans_a else 3) and batch_sizes.dim() == 1):
        return False
    if not (a.device == b.device and a.dtype in (torch.bfloat16, torch.float16, torch.float8_e4m3fn, torch.float8_e5m2)):
        return False
    hin = a.shape[1]
    hout = b.shape[1] if (trans_a or trans_b) else b.shape[2]
    experts = batch_sizes.shape[0]
    if trans_a:
        consistent = a.shape[0] == b.shape[0]
        out_shape = (experts, hin, hout)
    else:
        consistent = tuple(b.shape) == ((experts, hout, hin) if trans_b else (experts, hin, hout))
        out_shape = (a.shape[0], hout)
    if c is not None:
        consistent = (consistent and tuple(c.shape) == out_shape and c.device == a.device and
                      c.dtype == _output_dtype(a.dtype) and c.is_contiguous())
    if not consistent or hin == 0 or hout == 0 or a.shape[0] == 0:
        return False
    # (tensors that are not contiguous are rejected by the extension, as by the reference)
    if not (a.is_contiguous() and b.is_contiguous()):
        return False
    operands = (a, b) if c is None else (a, b, c)
    mult = 16 if a.element_size() == 1 else 8
    if hin % mult == 0 and hout % mult == 0 and all(t.data_ptr() % 16 == 0 for t in operands):
        return False
    # (otherwise the streaming kernels take these as they are)
    return not (a.element_size() == 2 and all(t.data_ptr() % 4 == 0 for t in operands) and hout % 2 == 0 and hin % 2 == 0)


def _padded(t, rows, cols):
    if t.shape[-2] == rows and t.shape[-1] == cols and t.data_ptr() % 16 == 0:
        return t
    return backend.pad_rows(t, rows, cols)


def _lined(t):
    """t, or a copy of it with zero-padded rows that the streaming kernels can read."""
    if t.shape[-1] % 8 == 0 and t.data_ptr() % 16 == 0:
        return t
    return backend.pad_rows(t, t.shape[-2], _padded_size(t.shape[-1], t.element_size()))


def _padded_call(a, b, c, batch_sizes, trans_a, trans_b):
    """gmm for operands that _needs_padding accepts."""
    hin = a.shape[1]
    hout = b.shape[1] if (trans_a or trans_b) else b.shape[2]
    if a.element_size() == 2:
        # (only what cannot be read as it is gets copied, and the result needs no copy)
        if c is None:
            c = _allocate_output(a, b, batch_sizes, trans_a, trans_b)
        backend.gmm_strided(_lined(a), _lined(b), c, batch_sizes, trans_a, trans_b and not trans_a, hin, hout)
        return c
    hin_p, hout_p = _padded_size(hin, a.element_size()), _padded_size(hout, a.element_size())
    a_p = _padded(a, a.shape[0], hin_p)
    if trans_a:
        b_p = _padded(b, b.shape[0], hout_p)
    else:
        b_p = _padded(b, hout_p, hin_p) if trans_b else _padded(b, hin_p, hout_p)
    return _padded_product(a_p, b_p, c, batch_sizes, trans_a, trans_b and not trans_a, hin, hout)


def _padded_product(a_p, b_p, c, batch_sizes, trans_a, trans_b, hin, hout):
    """The product of padded operands as an unpadded tensor: into c, or a new one where c is None."""
    hin_p, hout_p = a_p.shape[1], b_p.shape[1] if (trans_a or trans_b) else b_p.shape[2]
    dtype = _output_dtype(a_p.dtype)
    if trans_a:
        experts = batch_sizes.shape[0]
        if c is None:
            c = torch.empty(experts, hin, hout, dtype=dtype, device=a_p.device)
        whole = hin == hin_p and hout == hout_p and c.data_ptr() % 16 == 0
        c_p = c if whole else torch.empty(experts, hin_p, hout_p, dtype=dtype, device=a_p.device)   # all of it is written
    else:
        given = c is not None
        if c is None:
            c = torch.empty(a_p.shape[0], hout, dtype=dtype, device=a_p.device)
        # rows past sum(batch_sizes) are not written by the kernel and must keep what a given c holds
        if given or hout == hout_p:
            c_p = _padded(c, c.shape[0], hout_p)
        else:
            c_p = torch.empty(c.shape[0], hout_p, dtype=dtype, device=a_p.device)
    backend.gmm(a_p, b_p, c_p, batch_sizes, trans_a, trans_b)
    if c_p is not c:
        backend.unpad_rows(c_p, c)
    return c


def gradients(grad, a, b, batch_sizes, trans_b, want_a, want_b):
    """Both gradients of gmm(a, b, batch_sizes, trans_b=trans_b), each None where it is not wanted."""
    if want_a and want_b:
        both = backend.gmm_gradients(grad, a, b, batch_sizes, trans_b)   # (one launch)
        if both is not None:
            return both
    if want_a and want_b and _needs_padding(grad, b, None, batch_sizes, False, not trans_b) and \
            a.device == grad.device and a.dtype == grad.dtype and a.element_size() == 2 and a.is_contiguous() and \
            tuple(a.shape) == (grad.shape[0], b.shape[2 if trans_b else 1]):
        # (one padded copy of the gradient serves both products)
        return backend.gmm_gradients_strided(_lined(grad), _lined(a), _lined(b), batch_sizes, trans_b, a.shape[1], grad.shape[1])
    agrad = gmm(grad, b, batch_sizes, trans_a=False, trans_b=not trans_b) if want_a else None
    bgrad = None
    if want_b:
        lhs, rhs = (grad, a) if trans_b else (a, grad)
        bgrad = gmm(lhs, rhs, batch_sizes, trans_a=True, trans_b=False)
    return agrad, bgrad


def gmm(a, b, batch_sizes, trans_a=False, trans_b=False, c=None):
    out = backend.gmm_direct(a, b, batch_sizes, trans_a, trans_b, c)
    if out is not None:
        return out
    if c is None:
        _check_ranks(a, b, batch_sizes, trans_a, trans_b)
    if _needs_padding(a, b, c, batch_sizes, trans_a, trans_b):
        return _padded_call(a, b, c, batch_sizes, trans_a, trans_b)
    if c is None:
        c = _allocate_output(a, b, batch_sizes, trans_a, trans_b)
    backend.gmm(a, b, c, batch_sizes, trans_a, trans_b)
    return c


def gmm_indexed(a, b, batch_sizes, trans_a=False, trans_b=False, c=None, a_rows=None, b_rows=None,
                c_rows=None):
    """gmm with the permutation that sorts rows by expert fused in.  Not part of the reference's
    surface, whose `a` must already be sorted (grouped_gemm/ops.py:8).

    a_rows  int32 (tokens,): row r of the left operand is a[a_rows[r]] (a gather in the loads)
    b_rows  the same for the rows of b, with trans_a only
    c_rows  int32 (tokens,): row r of the product is stored to c[c_rows[r]] (a scatter in the
            stores; not with trans_a); needs `c`, whose other rows are left untouched

    Equal to gmm(a[a_rows], b, ...) and c[c_rows] = gmm(...), without the passes over a and c."""
    assert not (trans_a and trans_b)
    assert batch_sizes.ndim == 1, "Expected 1d tensor for batch_sizes"
    assert a.ndim == 2, "Expected 2d tensor for 'a'"
    assert b.ndim == (2 if trans_a else 3)
    if c is None:
        assert c_rows is None, "a scattered output needs the tensor to scatter into"
        tokens = a.shape[0] if a_rows is None else a_rows.shape[0]
        shape = ((batch_sizes.shape[0], a.shape[1], b.shape[1]) if trans_a else
                 (tokens, b.shape[1] if trans_b else b.shape[2]))
        c = torch.empty(*shape, device=a.device, dtype=_output_dtype(a.dtype))
    backend.gmm_indexed(a, b, c, batch_sizes, trans_a, trans_b, a_rows, b_rows, c_rows)
    return c


def gmm_swiglu(a, b, batch_sizes, trans_b=False, c=None, a_rows=None, c_rows=None):
    """silu(a_e @ gate_e) * (a_e @ up_e) per expert, the activation of a gated expert FFN computed in
    the epilogue of its first grouped GEMM.  b holds gate and up side by side: (experts, hidden_in,
    2 * hidden_out), or (experts, 2 * hidden_out, hidden_in) with trans_b, gate first.  Both products
    are accumulated and combined in fp32 and rounded once.  a_rows / c_rows as in gmm_indexed.
    Not part of the reference's surface (no epilogue hook: csrc/grouped_gemm.cu:255)."""
    assert batch_sizes.ndim == 1, "Expected 1d tensor for batch_sizes"
    assert a.ndim == 2, "Expected 2d tensor for 'a'"
    assert b.ndim == 3
    if c is None:
        assert c_rows is None, "a scattered output needs the tensor to scatter into"
        tokens = a.shape[0] if a_rows is None else a_rows.shape[0]
        c = torch.empty(tokens, (b.shape[1] if trans_b else b.shape[2]) // 2, device=a.device,
                        dtype=_output_dtype(a.dtype))
    backend.gmm_swiglu(a, b, c, batch_sizes, trans_b, a_rows, c_rows)
    return c


def accumulate_weight_gradient(a, b, batch_sizes, c):
    """c[e] += a_e^T @ b_e in fp32, for every expert e: the `trans_a` product of gmm added to
    an fp32 tensor (num_experts, a.shape[1], b.shape[1]) instead of written to a bf16 one.  Not
    part of the reference's surface (its kernels overwrite a bf16 output); for trainers that
    keep fp32 main gradients.  Returns c."""
    assert batch_sizes.ndim == 1, "Expected 1d tensor for batch_sizes"
    assert a.ndim == 2, "Expected 2d tensor for 'a'"
    assert b.ndim == 2, "Expected 2d tensor for 'b'"
    backend.accumulate_weight_gradient(a, b, c, batch_sizes)
    return c


def debug_schedule(batch_sizes, tokens, hidden_in, hidden_out, trans_a=False, trans_b=False,
                   device="cuda"):
    """Per-group table the on-device scheduler derives from `batch_sizes`: columns
    m, n, k, lda, ldb, ldc, a_off, b_off, c_off, first_tile, num_tiles, rows_used."""
    device = torch.device(device)
    if device.index is None:
        device = torch.device(device.type, torch.cuda.current_device())
    return backend.debug_schedule(batch_sizes, tokens, hidden_in, hidden_out, trans_a, trans_b, device)
