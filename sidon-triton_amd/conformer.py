"""The conformer layer's elementwise and convolution ops on the MI355X library.

Same names and argument meaning as src/sidon_triton/triton_encoder.py:

  * ``glu(h)`` (:127-133): h [R, 2C] fp16 -> h[:, :C] * sigmoid(h[:, C:]) fp16;
  * ``causal_dw_norm(g, batch, dwt, ln_w, ln_b, eps)`` (:163-181): g [B*T, C]
    fp16, dwt [K, C] fp32 -> silu(LN(causal depthwise conv)) fp16;
  * ``silu_(h)``: the in-place F.silu of the feed-forward modules (:498-499);
  * ``linear_silu(x, w, b)``: the feed-forward input projection and that SiLU
    in one kernel (``silu_(torch.addmm(b, x, w.t()))`` up to the GEMM's
    summation order; csrc/gemm.hip), for the shapes ``linear_silu_fits``
    accepts (N a multiple of 256, K of 64);

  * ``linear(x, w, b, out)`` and ``linear_glu(x, w)``: the plain projections
    and the pointwise conv's with its GLU (:500-505);
  * ``residual_gemm`` / ``residual_partials``: the projections into the fp32
    stream (:491-492), in place or as partial sums for the next norm;

plus ``glu_causal_dw_norm(h, ...)``, the two fused: it reads the pointwise
conv's output h [B*T, 2C] and forms g on the fly (bit-identical to
``causal_dw_norm(glu(h), ...)``, without the g round trip through HBM).

All launch on the current stream of the tensors' device through the C ABI of
include/sidon_encoder.h (csrc/conformer_ops.hip) and allocate only their
outputs (none when ``out`` is given), so they can be captured into HIP graphs.
"""

from __future__ import annotations

import ctypes

import torch
from torch.autograd import forward_ad

from . import _lib
from .flexrel import _check_device_tensor, _on_device, _stream_handle


def _fp16_rows(name, t, device, cols=None):
    _check_device_tensor(name, t, device)
    if t.dtype != torch.float16 or t.dim() != 2 or not t.is_contiguous():
        raise ValueError(f"{name} must be a contiguous float16 [R, C] tensor")
    if cols is not None and t.shape[1] != cols:
        raise ValueError(f"{name} must have {cols} columns (got {t.shape[1]})")


def glu(h: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    rows, c2 = h.shape
    if c2 % 2:
        raise ValueError("h must have an even number of columns")
    device = h.device
    _fp16_rows("h", h, device)
    c = c2 // 2
    if out is None:
        out = torch.empty(rows, c, device=device, dtype=h.dtype)
    else:
        _fp16_rows("out", out, device, c)
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_glu(h.data_ptr(), out.data_ptr(), rows, c, _stream_handle(device))
    _lib.check("sidon_glu", rc)
    return out


def silu_(h: torch.Tensor) -> torch.Tensor:
    """h = h * sigmoid(h) in place (fp16, any shape, contiguous)."""
    device = h.device
    _check_device_tensor("h", h, device)
    if h.dtype != torch.float16 or not h.is_contiguous():
        raise ValueError("h must be a contiguous float16 tensor")
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_silu(h.data_ptr(), h.numel(), _stream_handle(device))
    _lib.check("sidon_silu", rc)
    return h


def _dw(src, glu_input, batch, dwt, ln_w, ln_b, eps, out):
    rows, width = src.shape
    c = width // 2 if glu_input else width
    device = src.device
    _fp16_rows("h" if glu_input else "g", src, device)
    if rows % batch:
        raise ValueError(f"{rows} rows do not split into {batch} items")
    for name, t, shape in (("dwt", dwt, None), ("ln_w", ln_w, (c,)), ("ln_b", ln_b, (c,))):
        _check_device_tensor(name, t, device)
        if t.dtype != torch.float32 or not t.is_contiguous():
            raise ValueError(f"{name} must be a contiguous float32 tensor")
        if shape is not None and tuple(t.shape) != shape:
            raise ValueError(f"{name} must be [{c}]")
    if dwt.dim() != 2 or dwt.shape[1] != c:
        raise ValueError(f"dwt must be [K, {c}]")
    if out is None:
        out = torch.empty(rows, c, device=device, dtype=torch.float16)
    else:
        _fp16_rows("out", out, device, c)
        if out.shape[0] != rows:
            raise ValueError("out must have the input's rows")
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_causal_dw_norm(src.data_ptr(), int(glu_input), dwt.data_ptr(), ln_w.data_ptr(),
                                      ln_b.data_ptr(), ctypes.c_float(float(eps)), out.data_ptr(), batch,
                                      rows // batch, c, dwt.shape[0], _stream_handle(device))
    _lib.check("sidon_causal_dw_norm", rc)
    return out


def causal_dw_norm(g: torch.Tensor, batch: int, dwt: torch.Tensor, ln_w: torch.Tensor, ln_b: torch.Tensor,
                   eps: float, out: torch.Tensor | None = None) -> torch.Tensor:
    """g [B*T, C] fp16 -> silu(LN(sum_k dwt[k] * g[t + k - (K-1)])) [B*T, C] fp16
    (zero left padding per item; dwt [K, C] fp32, ln_w / ln_b [C] fp32)."""
    return _dw(g, False, batch, dwt, ln_w, ln_b, eps, out)


def glu_causal_dw_norm(h: torch.Tensor, batch: int, dwt: torch.Tensor, ln_w: torch.Tensor, ln_b: torch.Tensor,
                       eps: float, out: torch.Tensor | None = None) -> torch.Tensor:
    """causal_dw_norm(glu(h), ...) in one pass: h [B*T, 2C] fp16."""
    return _dw(h, True, batch, dwt, ln_w, ln_b, eps, out)


def linear_silu_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether ``linear_silu`` takes x [M, K] and w [N, K]."""
    return bool(_lib.load().sidon_gemm_bias_act_fits(x.shape[0], w.shape[0], w.shape[1])) and x.shape[1] == w.shape[1]


def linear_silu_preferred(rows: int, n: int, k: int, device=None) -> bool:
    """Whether ``linear_silu`` is expected to beat ``linear_silu_lt`` and
    ``silu_(torch.addmm(...))`` for x [rows, k], w [n, k] on ``device`` (past
    ``linear_silu_lt``'s own kernel, where 320 x 256 tiles would fill >= 4/5 of
    the CUs in every round; at n = 4096, k = 1024 that is rows > 3840 on 256 CUs,
    of which those up to 4096 are 10% faster on ``linear_silu_lt``)."""
    with _on_device(device):
        return bool(_lib.load().sidon_gemm_bias_act_preferred(rows, n, k))


def _linear_args(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None, out: torch.Tensor | None):
    device = x.device
    for name, t in (("x", x), ("w", w)):
        _check_device_tensor(name, t, device)
        if t.dtype != torch.float16 or t.dim() != 2 or t.stride(1) != 1:
            raise ValueError(f"{name} must be a float16 [rows, K] tensor with K contiguous")
    rows, k = x.shape
    n = w.shape[0]
    if w.shape[1] != k:
        raise ValueError(f"x has {k} columns, w {w.shape[1]}")
    if b is not None:
        _check_device_tensor("b", b, device)
        if b.dtype != torch.float16 or tuple(b.shape) != (n,) or not b.is_contiguous():
            raise ValueError(f"b must be a contiguous float16 [{n}] tensor")
    if out is None:
        out = torch.empty(rows, n, device=device, dtype=torch.float16)
    else:
        _check_device_tensor("out", out, device)
        if out.dtype != torch.float16 or tuple(out.shape) != (rows, n) or out.stride(1) != 1:
            raise ValueError(f"out must be a float16 [{rows}, {n}] tensor with rows contiguous")
    return rows, n, k, out


def linear_silu(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None, out: torch.Tensor | None = None,
                act: bool = True) -> torch.Tensor:
    """silu(fp16(x . w^T + b)) [M, N] fp16 for x [M, K] and w [N, K] fp16
    (rows K-contiguous), b [N] fp16 or None; act=False leaves out the SiLU."""
    device = x.device
    rows, n, k, out = _linear_args(x, w, b, out)
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_gemm_bias_act(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                                     None if b is None else b.data_ptr(), out.data_ptr(), out.stride(0), rows, n, k,
                                     1 if act else 0, _stream_handle(device))
    _lib.check("sidon_gemm_bias_act", rc)
    return out


def linear_silu_lt(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor | None, out: torch.Tensor | None = None,
                   act: bool = True) -> torch.Tensor:
    """silu(x . w^T + b) [M, N] fp16 with the bias and SiLU in the GEMM's
    epilogue (fp32 sum + bias, SiLU in fp32, one rounding to fp16), for
    x [M, K] and w [N, K] fp16 (rows K-contiguous), b [N] fp16 or None;
    act=False leaves out the SiLU.  On this library's tiled kernel where
    ``sidon_gemm_half_preferred`` and the alignment allow, else on hipBLASLt,
    whose first call on a device must not run during stream capture."""
    device = x.device
    rows, n, k, out = _linear_args(x, w, b, out)
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_gemm_lt_act(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                                   None if b is None else b.data_ptr(), out.data_ptr(), out.stride(0), rows, n, k,
                                   1 if act else 0, _stream_handle(device))
    _lib.check("sidon_gemm_lt_act", rc)
    return out


def tile_operand(t: torch.Tensor) -> bool:
    """Whether the tiled GEMM kernel's 16-byte copies take t [rows, K] as an
    operand: fp16, K contiguous, rows apart and 16-byte aligned."""
    return (t.dtype == torch.float16 and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) >= t.shape[1]
            and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0)


def plain(*tensors: torch.Tensor) -> bool:
    """Whether a kernel may stand in for a torch call with ``out=`` on these:
    no subclass of its own behaviour, and nothing that autograd, in reverse or
    forward mode, would follow (torch refuses ``out=`` there)."""
    if any(type(t) not in (torch.Tensor, torch.nn.Parameter) for t in tensors):
        return False
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return False
    return (getattr(forward_ad, "_current_level", 0) < 0
            or all(forward_ad.unpack_dual(t).tangent is None for t in tensors))


def linear(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """out = x . w^T + b, fp16 with fp32 sums: this library's GEMM kernel up to
    the sizes where it beats the library, for operands as it reads them
    (``sidon_gemm_half_takes``), else torch.addmm (any strides, a broadcast b).
    x [M, K], w [N, K], out [M, N]."""
    own = (plain(x, w, b, out) and tile_operand(x) and tile_operand(w) and x.shape[1] == w.shape[1]
           and b.dtype == torch.float16 and tuple(b.shape) == (w.shape[0],) and b.is_contiguous()
           and tuple(out.shape) == (x.shape[0], w.shape[0]) and tile_operand(out)
           and _lib.load().sidon_gemm_half_takes(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), b.data_ptr(),
                                                 out.data_ptr(), out.stride(0), *out.shape, x.shape[1]))
    if own:
        return linear_silu_lt(x, w, b, out=out, act=False)
    return torch.addmm(b, x, w.t(), out=out)


def linear_glu_fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether ``linear_glu`` takes x [M, K] and w [2C, K] (each spanning less
    than 4 GiB)."""
    return (w.shape[0] % 64 == 0 and w.shape[1] % 64 == 0 and x.shape[1] == w.shape[1] and tile_operand(x)
            and tile_operand(w) and all(2 * t.shape[0] * t.stride(0) < 1 << 32 for t in (x, w)))


def linear_glu(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """``glu(x . w^T)`` in one kernel (src/sidon_triton/triton_encoder.py:504-505):
    x [M, K] and w [2C, K] fp16 with K contiguous -> [M, C] fp16, the products
    rounded to fp16 in front of the GLU as a separate GEMM stores them."""
    device = x.device
    for name, t in (("x", x), ("w", w)):
        _check_device_tensor(name, t, device)
        if t.dtype != torch.float16 or t.dim() != 2 or t.stride(1) != 1:
            raise ValueError(f"{name} must be a float16 [rows, K] tensor with K contiguous")
    rows, k = x.shape
    if w.shape[1] != k or w.shape[0] % 2:
        raise ValueError(f"x is {tuple(x.shape)}, w {tuple(w.shape)}")
    c = w.shape[0] // 2
    if out is None:
        out = torch.empty(rows, c, device=device, dtype=torch.float16)
    else:
        _check_device_tensor("out", out, device)
        if out.dtype != torch.float16 or tuple(out.shape) != (rows, c) or out.stride(1) != 1:
            raise ValueError(f"out must be a float16 [{rows}, {c}] tensor with rows contiguous")
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_gemm_glu(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0),
                                rows, c, k, _stream_handle(device))
    _lib.check("sidon_gemm_glu", rc)
    return out


def residual_gemm_fits(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether ``residual_gemm`` takes a [M, K], w [N, K] into x [M, N]."""
    return (bool(_lib.load().sidon_gemm_res_fits(a.shape[0], w.shape[0], w.shape[1])) and a.shape[1] == w.shape[1]
            and tuple(x.shape) == (a.shape[0], w.shape[0]))


def residual_gemm_preferred(rows: int, n: int, k: int, device=None) -> bool:
    """Whether ``residual_gemm`` is expected to beat torch.addmm for a
    [rows, k], w [n, k] on ``device`` (up to 5 * 2^20 outputs; in a graph
    torch.addmm is 2-3 us faster up to 2^18 outputs where k > 2048)."""
    with _on_device(device):
        return bool(_lib.load().sidon_gemm_res_preferred(rows, n, k))


def residual_splits(rows: int, n: int, k: int, device=None, part: bool = True) -> int:
    """K ranges of ``residual_partials`` for a [rows, k], w [n, k]: 2 to 8, or 1
    where the in-place ``residual_gemm`` is the better call, or 0 where
    torch.addmm is.  ``part`` False: the caller has no buffer for partial sums,
    so 1 or 0.  Depends on these and the device alone."""
    lib = _lib.load()
    with _on_device(device):
        splits = int(lib.sidon_gemm_part_splits(rows, n, k)) if part else 0
        return splits if splits > 1 else int(lib.sidon_gemm_res_preferred(rows, n, k))


def partial_values(rows: int, n: int) -> int:
    """fp32 values that hold the partial sums of any call of up to ``rows`` rows."""
    return int(_lib.load().sidon_gemm_part_rows(rows)) * n


def _residual_operands(a: torch.Tensor, w: torch.Tensor, device: torch.device):
    for name, t in (("a", a), ("w", w)):
        _check_device_tensor(name, t, device)
        if t.dtype != torch.float16 or t.dim() != 2 or t.stride(1) != 1:
            raise ValueError(f"{name} must be a float16 [rows, K] tensor with K contiguous")
    if w.shape[1] != a.shape[1]:
        raise ValueError(f"a has {a.shape[1]} columns, w {w.shape[1]}")
    return a.shape[0], w.shape[0], a.shape[1]


def residual_partials(a: torch.Tensor, w: torch.Tensor, part: torch.Tensor) -> torch.Tensor:
    """a . w^T [M, N] as partial sums over ``residual_splits`` K ranges, for
    ``encoder_block.res_norm_parts`` to add to the stream: a [M, K] and w [N, K]
    fp16 with K contiguous, part a contiguous fp32 buffer (``partial_values``).
    Returns the [splits, M, N] view of ``part`` that holds them."""
    device = a.device
    rows, n, k = _residual_operands(a, w, device)
    _check_device_tensor("part", part, device)
    if part.dtype != torch.float32 or not part.is_contiguous():
        raise ValueError("part must be a contiguous float32 tensor")
    lib = _lib.load()
    with _on_device(device):
        splits = lib.sidon_gemm_part_splits(rows, n, k)
        rc = lib.sidon_gemm_part(a.data_ptr(), a.stride(0), w.data_ptr(), w.stride(0), part.data_ptr(), part.numel(),
                                 rows, n, k, _stream_handle(device))
    _lib.check("sidon_gemm_part", rc)
    return part.view(-1)[:splits * rows * n].view(splits, rows, n)


def residual_gemm(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x += a . w^T in place: x [M, N] fp32 (the residual stream), a [M, K]
    and w [N, K] fp16 with K contiguous -- the
    ``torch.addmm(x, a, w.t(), out_dtype=torch.float32, out=x)`` of the
    reference's res() (src/sidon_triton/triton_encoder.py:491-492).  Takes no
    memory but x; a caller with a buffer for partial sums has short streams
    faster through ``residual_partials`` and ``encoder_block.res_norm_parts``."""
    device = x.device
    rows, n, k = _residual_operands(a, w, device)
    _check_device_tensor("x", x, device)
    if x.dtype != torch.float32 or tuple(x.shape) != (rows, n) or x.stride(1) != 1:
        raise ValueError(f"x must be a float32 [{rows}, {n}] tensor with rows contiguous")
    lib = _lib.load()
    with _on_device(device):
        rc = lib.sidon_gemm_res(a.data_ptr(), a.stride(0), w.data_ptr(), w.stride(0), x.data_ptr(), x.stride(0),
                                rows, n, k, _stream_handle(device))
    _lib.check("sidon_gemm_res", rc)
    return x
