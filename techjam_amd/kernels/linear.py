"""Dense layers of the encoder block on the split-bf16 HIP kernels.

They do the arithmetic of hipBLASLt's fast float32 mode (operands split into
two bf16 parts, three products, fp32 accumulation; same error against 64
bits), so they are used only where a float32 product would run in that mode
(:func:`fast_float32_matmul`) and, as a raw kernel call records no graph, only
while gradients are off. Each function returns ``None`` for what it does not
take or is not faster at, and the caller then uses the library.
"""

from __future__ import annotations

from typing import Optional, Sequence, Tuple

import torch

from . import _lib
from .attention import _stream_ptr

#: Width of the layers the one-pass kernels take.
NARROW = 128
#: Multiply-adds up to which the small-tile kernel is used, and its depth (at
#: K = 1024 and 256 x 256 the library takes 9.5 us, this 10.2). One product, us by the library / here, replayed as graphs: 32 x 256 x
#: 256 11.0 / 4.4, 256 x 256 x 256 26.0 / 4.5, 256 x 512 x 512 7.5 / 6.4, 1200
#: x 128 x 512 7.5 / 6.5; past the line 1200 x 512 x 512 11.2 / 17.2.
ROWS_MAX_WORK = 1 << 26
ROWS_MAX_K = 512
#: Tokens from which the one-pass kernels beat a product and the passes after
#: it, and up to which the shorter one does (us, library + passes / here:
#: residual + norm 16 384 tokens 16.4 / 16.4, 65 536 38 / 31, 262 144 146 / 155;
#: FFN 30 / 38, 66 / 41, 249 / 205): below, one tile's latency is all there is.
NARROW_MIN_TOKENS = 24576
NARROW_RESIDUAL_MAX_TOKENS = 131072


#: The setting float32 GEMMs on the GPU obey (``torch.backends.cuda.matmul.
#: fp32_precision``, at a third of that property's cost); ``None`` on a torch
#: without it.
_fp32_precision = getattr(torch._C, "_get_fp32_precision_getter", None)


def fast_float32_matmul() -> bool:
    """Whether a float32 product on the GPU runs on split bf16 operands.

    That is hipBLASLt's fast mode: the other BLAS backends compute in plain
    float32 at any setting (256 x 256 x 256: 2.9e-7 of error, split 4.4e-6).
    ``torch.get_float32_matmul_precision()`` does not tell -- it still says
    "high" after ``torch.backends.cuda.matmul.fp32_precision`` was set to
    "ieee", and raises where the two disagree the other way.
    """
    if _fp32_precision is None:
        fast = torch.get_float32_matmul_precision() != "highest"
    else:
        fast = _fp32_precision("cuda", "matmul") == "tf32"
    return fast and torch._C._get_blas_preferred_backend() == torch._C._BlasBackend.Cublaslt


def _usable(x: torch.Tensor, *params: torch.Tensor) -> bool:
    if (not x.is_cuda or x.dtype != torch.float32 or torch.is_grad_enabled()
            or not fast_float32_matmul() or not x.is_contiguous() or x.data_ptr() % 16
            or torch.is_autocast_enabled("cuda")):  # the product would give the autocast type
        return False
    dev = x.device
    for p in params:
        if (p is None or p.dtype != torch.float32 or p.device != dev or not p.is_contiguous() or p.data_ptr() % 16):
            return False
    return True


def projections(x: torch.Tensor, weights: Sequence[torch.Tensor], bias: Optional[torch.Tensor] = None,
                act: Optional[str] = None) -> Optional[Tuple[torch.Tensor, ...]]:
    """``x @ w.T`` for up to three weights of one shape in one launch, or
    ``act(x @ w.T + bias)`` for one (``act`` "gelu" or "relu")."""
    n, k = weights[0].shape
    if x.numel() * n * len(weights) <= ROWS_MAX_WORK:
        if n & 31 or k & 63 or k > ROWS_MAX_K:
            return None
        narrow = 0
    elif n == NARROW and k == NARROW and act is None:
        narrow = 1
    else:
        return None
    m = x.numel() // k
    if (x.shape[-1] != k or m == 0 or not _usable(x, *weights, *(() if bias is None else (bias,)))
            or any(w.shape != (n, k) for w in weights) or (bias is not None and bias.shape != (n,))):
        return None  # the kernel reads n values of the bias
    outs = [torch.empty(*x.shape[:-1], n, dtype=x.dtype, device=x.device) for _ in weights]
    ptrs = [w.data_ptr() for w in weights] + [None] * (3 - len(weights))
    optr = [o.data_ptr() for o in outs] + [None] * (3 - len(weights))
    code = _lib.lib().tj_linear(x.data_ptr(), *ptrs, *optr, m, n, k, None if bias is None else bias.data_ptr(),
                                {None: 0, "gelu": 1, "relu": 2}[act], narrow, _stream_ptr(x.device))
    _lib.check(code, "tj_linear")
    return tuple(outs)


def _residual_ok(x, resid, bias, valid_len, norm, params) -> bool:
    return (x.ndim == 3 and x.shape[-1] == NARROW and x.numel() > 0 and resid.shape == x.shape
            and all(p is not None and p.shape == (NARROW, NARROW) for p in params)
            and bias is not None and bias.shape == (NARROW,)
            and isinstance(norm, torch.nn.LayerNorm) and tuple(norm.normalized_shape) == (NARROW,)
            and norm.weight is not None and norm.bias is not None
            and _usable(x, resid, bias, norm.weight, norm.bias, *params)
            and (valid_len is None or (valid_len.dtype == torch.int32 and valid_len.shape == (x.shape[0],)
                                       and valid_len.device == x.device and valid_len.is_contiguous())))


def residual_norm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor, resid: torch.Tensor,
                  valid_len: Optional[torch.Tensor], mode: int, norm: torch.nn.LayerNorm,
                  zero_padded_norm: bool = False):
    """``kernels.elementwise.bias_residual_layernorm`` of ``y = x @ weight.T``
    in one pass, for layers of width 128: ``(out, norm(out))``."""
    if (not NARROW_MIN_TOKENS <= x.numel() // NARROW <= NARROW_RESIDUAL_MAX_TOKENS
            or not _residual_ok(x, resid, bias, valid_len, norm, (weight,))):
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
             norm: torch.nn.LayerNorm, zero_padded_norm: bool = False):
    """The same with ``y = act(x @ w_in.T + b_in) @ w_out.T``: the FFN half of
    a block of width 128 whose hidden layer is 128 wide too."""
    if (x.numel() // NARROW < NARROW_MIN_TOKENS
            or not _residual_ok(x, resid, bias, valid_len, norm, (w_in, w_out)) or b_in is None
            or b_in.shape != (NARROW,) or not _usable(x, b_in)):
        return None
    out, ln = torch.empty_like(resid), torch.empty_like(resid)
    code = _lib.lib().tj_narrow_ffn_norm(
        x.data_ptr(), w_in.data_ptr(), b_in.data_ptr(), {"gelu": 1, "relu": 2}[act], w_out.data_ptr(),
        bias.data_ptr(), resid.data_ptr(), out.data_ptr(), x.numel() // NARROW, x.shape[1],
        None if valid_len is None else valid_len.data_ptr(), mode, norm.weight.data_ptr(), norm.bias.data_ptr(),
        ln.data_ptr(), float(norm.eps), int(bool(zero_padded_norm)), _stream_ptr(x.device))
    _lib.check(code, "tj_narrow_ffn_norm")
    return out, ln
