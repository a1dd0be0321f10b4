"""Dense layers of the encoder block on the split-bf16 HIP kernels.

They do the arithmetic of hipBLASLt's fast float32 mode (operands split into
two bf16 parts, three products, fp32 accumulation; same error against 64
bits), so they are used only where a float32 product would run in that mode
and, as a raw kernel call records no graph, only while gradients are off
(:func:`split_products_allowed`, which a caller of several of them asks once
and hands on as ``allowed``). Each function returns ``None`` for what it does
not take or is not faster at, and the caller then uses the library.
"""

from __future__ import annotations

from typing import Optional, Sequence, Tuple

import torch

from . import _lib
from .attention import _stream_ptr

#: Width of the layers the one-pass kernels take.
NARROW = 128
#: Multiply-adds up to which the small-tile kernel is used, and its depth (at
#: K = 1024 and 256 x 256 the library takes 9.5 us, this 10.2). One product, us
#: by the library / here, replayed as graphs: 32 x 256 x 256 11.0 / 4.4, 256 x
#: 256 x 256 26.0 / 4.5, 256 x 512 x 512 7.5 / 6.4, 1200 x 128 x 512 7.5 / 6.5;
#: past the line 1200 x 512 x 512 11.2 / 17.2. Called one after another, a
#: lone product is bound by its call, 19.2 us by the library and 8.7 here, also
#: where its kernel alone is behind: 4 x 1024 x 256 3.8 / 4.1, 16 x 512 x 512
#: 4.5 / 6.0, 8192 x 128 x 64 5.1 / 6.1, and at width 128 from 4098 tokens (5.8
#: / 7.7) to 24 576 (9.3 / 9.5). A replayed forward gives up to 2 us there.
ROWS_MAX_WORK = 1 << 26
ROWS_MAX_K = 512
#: Tokens from which the one-pass kernels beat a product and the passes after
#: it, and up to which the shorter one does (us, library + passes / here,
#: replayed: residual + norm 16 384 tokens 17.1 / 17.1, 24 576 21.4 / 18.2,
#: 98 304 57 / 45, 122 880 72 / 55, 131 072 72 / 75, 262 144 151 / 161; FFN
#: 30.7 / 30.7, 34 / 32, 95 / 61, 125 / 78 at 131 072, 259 / 166): below, one
#: tile's latency is all there is; above, the sum in a buffer of its own takes
#: the four tensors past the memory-side cache.
NARROW_MIN_TOKENS = 24576
NARROW_RESIDUAL_MAX_TOKENS = 122880

_ACT = {None: 0, "gelu": 1, "relu": 2}
_NONE = (None, None, None)
_HIPBLASLT = torch._C._BlasBackend.Cublaslt.value


def split_products_allowed() -> bool:
    """Whether a float32 ``F.linear`` on the GPU would run here and now on
    split bf16 operands, with a float32 result and no graph to record.

    The split form is hipBLASLt's fast mode: the other BLAS backends compute in
    plain float32 at any setting (256 x 256 x 256: 2.9e-7 of error, split
    4.4e-6). ``torch.get_float32_matmul_precision()`` does not tell the mode --
    it still says "high" after ``torch.backends.cuda.matmul.fp32_precision`` was
    set to "ieee", and raises where the two disagree the other way.
    """
    if torch.is_grad_enabled() or torch.is_autocast_enabled():  # autocast: the result has its type
        return False
    try:
        fast = torch._C._get_cublas_allow_tf32()  # a quarter of the cost of fp32_precision
    except RuntimeError:  # the older and the newer setting disagree; the GEMMs obey the newer
        fast = torch.backends.cuda.matmul.fp32_precision == "tf32"
    return fast and torch._C._get_blas_preferred_backend().value == _HIPBLASLT


def _usable(allowed: Optional[bool], x: torch.Tensor, *params: torch.Tensor) -> Optional[list]:
    """The addresses of ``x`` and ``params`` if the kernels may run on them."""
    if not x.is_cuda or not (split_products_allowed() if allowed is None else allowed):
        return None
    dev, f32, ptrs = x.get_device(), torch.float32, []
    for t in (x, *params):
        if t is None or t.dtype != f32 or t.get_device() != dev or not t.is_contiguous():
            return None
        p = t.data_ptr()
        if p & 15:
            return None
        ptrs.append(p)
    return ptrs


def projections(x: torch.Tensor, weights: Sequence[torch.Tensor], bias: Optional[torch.Tensor] = None,
                act: Optional[str] = None, allowed: Optional[bool] = None) -> Optional[Tuple[torch.Tensor, ...]]:
    """``x @ w.T`` for up to three weights of one shape in one launch, or
    ``act(x @ w.T + bias)`` for one (``act`` "gelu" or "relu")."""
    # Plain statements: small blocks are bound by this function's own cost.
    w_shape, n_w, size = weights[0].shape, len(weights), x.numel()
    n, k = w_shape
    if size * n * n_w <= ROWS_MAX_WORK:
        if n & 31 or k & 63 or k > ROWS_MAX_K:
            return None
        narrow = 0
    elif n == NARROW and k == NARROW and act is None:
        narrow = 1
    else:
        return None
    shape = x.shape
    if shape[-1] != k or size == 0:
        return None
    for w in weights:
        if w.shape != w_shape:
            return None
    if bias is None:
        ptrs = _usable(allowed, x, *weights)
    elif bias.shape == (n,):  # the kernel reads n values
        ptrs = _usable(allowed, x, *weights, bias)
    else:
        return None
    if ptrs is None:
        return None
    out_shape = (*shape[:-1], n)
    outs = [x.new_empty(out_shape) for _ in weights]
    pad = _NONE[n_w:]
    code = _lib.lib().tj_linear(*ptrs[:1 + n_w], *pad, *[o.data_ptr() for o in outs], *pad, size // k, n, k,
                                None if bias is None else ptrs[-1], _ACT[act], narrow, _stream_ptr(x.device))
    if code:
        _lib.check(code, "tj_linear")
    return tuple(outs)


def _residual_ok(allowed, x, resid, weights, biases, valid_len, norm) -> bool:
    return (x.ndim == 3 and x.shape[-1] == NARROW and x.numel() > 0 and resid.shape == x.shape
            and all(w is not None and w.shape == (NARROW, NARROW) for w in weights)
            and all(b is not None and b.shape == (NARROW,) for b in biases)
            and isinstance(norm, torch.nn.LayerNorm) and tuple(norm.normalized_shape) == (NARROW,)
            and norm.weight is not None and norm.bias is not None
            and _usable(allowed, x, resid, norm.weight, norm.bias, *weights, *biases) is not None
            and (valid_len is None or (valid_len.dtype == torch.int32 and valid_len.shape == (x.shape[0],)
                                       and valid_len.device == x.device and valid_len.is_contiguous())))


def residual_norm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, resid: torch.Tensor,
                  valid_len: Optional[torch.Tensor], mode: int, norm: torch.nn.LayerNorm,
                  zero_padded_norm: bool = False, allowed: Optional[bool] = None):
    """``kernels.elementwise.bias_residual_layernorm`` of ``y = x @ weight.T``
    in one pass, for layers of width 128: ``(out, norm(out))``."""
    if (not NARROW_MIN_TOKENS <= x.numel() // NARROW <= NARROW_RESIDUAL_MAX_TOKENS
            or not _residual_ok(allowed, x, resid, (weight,), (bias,), valid_len, norm)):
        return None
    out, ln = torch.empty_like(resid), torch.empty_like(resid)
    code = _lib.lib().tj_narrow_residual_norm(
        x.data_ptr(), weight.data_ptr(), bias.data_ptr(), resid.data_ptr(), out.data_ptr(), x.numel() // NARROW,
        x.shape[1], None if valid_len is None else valid_len.data_ptr(), mode, norm.weight.data_ptr(),
        norm.bias.data_ptr(), ln.data_ptr(), float(norm.eps), int(bool(zero_padded_norm)), _stream_ptr(x.device))
    _lib.check(code, "tj_narrow_residual_norm")
    return out, ln


def ffn_norm(x: torch.Tensor, w_in: torch.Tensor, b_in: torch.Tensor, act: str, w_out: torch.Tensor,
             bias: torch.Tensor, resid: torch.Tensor, valid_len: Optional[torch.Tensor], mode: int,
             norm: torch.nn.LayerNorm, zero_padded_norm: bool = False, allowed: Optional[bool] = None):
    """The same with ``y = act(x @ w_in.T + b_in) @ w_out.T``: the FFN half of
    a block of width 128 whose hidden layer is 128 wide too."""
    if (x.numel() // NARROW < NARROW_MIN_TOKENS
            or not _residual_ok(allowed, x, resid, (w_in, w_out), (b_in, bias), valid_len, norm)):
        return None
    out, ln = torch.empty_like(resid), torch.empty_like(resid)
    code = _lib.lib().tj_narrow_ffn_norm(
        x.data_ptr(), w_in.data_ptr(), b_in.data_ptr(), _ACT[act], w_out.data_ptr(),
        bias.data_ptr(), resid.data_ptr(), out.data_ptr(), x.numel() // NARROW, x.shape[1],
        None if valid_len is None else valid_len.data_ptr(), mode, norm.weight.data_ptr(), norm.bias.data_ptr(),
        ln.data_ptr(), float(norm.eps), int(bool(zero_padded_norm)), _stream_ptr(x.device))
    _lib.check(code, "tj_narrow_ffn_norm")
    return out, ln
