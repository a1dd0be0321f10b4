"""Transformer encoder skeleton whose attention runs on the HIP kernels.

Same module tree, parameter names and construction order as the reference
model (``torch_transformer_benchmark.py:29-172``), so the harness's strict
``load_state_dict`` works unchanged and a seeded construction gives the same
weights. Only the attention module differs: ``HipSelfAttention`` projects with
``Linear`` (an ``nn.Linear`` whose bias add stays outside the GEMM when the
fast float32 matmul mode is on) and calls the gfx950 attention kernel through
the C ABI instead of materialising a score tensor. Without gradients the
projections run bias-free, small and 128-wide ones on the kernels of
``kernels/linear.py``, the rest on the BLAS library (hipBLASLt by default).
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F

from .kernels.attention import scaled_dot_product_attention
from .kernels.elementwise import NORM_WIDTHS
from .kernels.linear import ffn_norm, projections, residual_norm, split_products_allowed


ACTIVATIONS = ("gelu", "relu")


@dataclass(frozen=True)
class TransformerConfig:
    """Static model shape; field names follow ``torch_transformer_benchmark.py:29-56``.

    ``norm_first`` and ``activation`` select the block: the reference model is
    pre-norm with exact GELU (the defaults); ``norm_first=False,
    activation="relu"`` is the post-norm / ReLU block of
    ``torch.nn.TransformerEncoderLayer(norm_first=False, activation="relu")``,
    the wording some benchmark configurations are stated in. Config objects
    without these fields (the reference harness's own) mean the defaults.
    """

    batch_size: int
    seq_len: int
    d_model: int
    num_heads: int
    ffn_dim: int
    num_layers: int
    causal: bool
    norm_first: bool = True
    activation: str = "gelu"

    def validate(self) -> None:
        for name in ("batch_size", "seq_len", "d_model", "num_heads", "ffn_dim", "num_layers"):
            if getattr(self, name) <= 0:
                raise ValueError(f"{name} must be positive")
        if self.d_model % self.num_heads:
            raise ValueError(
                f"d_model ({self.d_model}) must be divisible by num_heads ({self.num_heads})"
            )
        if self.activation not in ACTIVATIONS:
            raise ValueError(f"activation must be one of {ACTIVATIONS}, not {self.activation!r}")


def block_variant(config) -> Tuple[bool, str]:
    """``(norm_first, activation)`` of a config; the reference's block when the
    config does not say."""
    norm_first = bool(getattr(config, "norm_first", True))
    activation = getattr(config, "activation", "gelu")
    if activation not in ACTIVATIONS:
        raise ValueError(f"activation must be one of {ACTIVATIONS}, not {activation!r}")
    return norm_first, activation


def config_key(config) -> tuple:
    """The 7-tuple route key ``(B, S, d_model, H, ffn, causal, layers)`` (``src/dispatcher.py:74-83``)."""
    return (config.batch_size, config.seq_len, config.d_model, config.num_heads,
            config.ffn_dim, config.causal, config.num_layers)


def _linear_f32(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``F.linear`` on torch's configured BLAS backend (no process-global
    state is changed per call)."""
    return F.linear(x, weight, bias)


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    """``F.linear``; when float32 matmuls may use the faster hipBLASLt mode
    (``torch.get_float32_matmul_precision() != "highest"``, the reference
    harness's validated setting) the bias is added after a bias-free GEMM,
    because the fused-bias GEMM ignores that mode on this stack (16384x1024 by
    1024x3072: 0.72 ms fused either way, 0.29 ms bias-free in the fast mode)."""
    if bias is None or x.device.type != "cuda" or torch.get_float32_matmul_precision() == "highest":
        return _linear_f32(x, weight, bias)
    y = _linear_f32(x, weight)
    y += bias
    return y


def fp16_weight(owner: nn.Module, key: str, weight: torch.Tensor) -> torch.Tensor:
    """Rounded fp16 copy of ``weight``, cached on ``owner`` and rebuilt
    whenever the weight is replaced or modified in place."""
    try:
        version = weight._version
    except RuntimeError:
        # An inference tensor carries no version counter, so an in-place
        # refill could not be seen: convert on every call instead of caching.
        return weight.detach().to(torch.float16)
    cache = owner.__dict__.setdefault("_fp16_weights", {})
    tag = (weight.data_ptr(), version, weight.device, tuple(weight.shape))
    hit = cache.get(key)
    if hit is None or hit[0] != tag:
        hit = (tag, weight.detach().to(torch.float16))
        cache[key] = hit
    return hit[1]


def project(x: torch.Tensor, weight: torch.Tensor, owner: nn.Module, key: str,
            out_dtype: Optional[torch.dtype] = None, allowed: Optional[bool] = None) -> torch.Tensor:
    """Bias-free ``x @ weight.T``. A float32 ``x`` runs the float32 GEMM
    (``allowed``: what :func:`split_products_allowed` says, if the caller
    asked); a float16 ``x`` runs on fp16 operands (the weight's cached fp16
    copy) with fp32 accumulation, its result in ``out_dtype`` (default float16)."""
    if x.dtype != torch.float16:
        own = projections(x, (weight,), allowed=allowed)
        return _linear_f32(x, weight) if own is None else own[0]
    w16 = fp16_weight(owner, key, weight)
    if out_dtype in (None, torch.float16):
        return F.linear(x, w16)
    flat = x.reshape(-1, x.shape[-1])
    return torch.mm(flat, w16.t(), out_dtype=out_dtype).view(*x.shape[:-1], w16.shape[0])


class Linear(nn.Linear):
    """``nn.Linear`` with the same parameters and state-dict names whose
    forward is :func:`linear`."""

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return linear(x, self.weight, self.bias)


class HipSelfAttention(nn.Module):
    """Multi-head self-attention: Linear projections + the HIP exact kernel.

    ``valid_len`` (int32 ``[B]`` on the device) carries a right-padded mask to
    the kernel: keys past the length are excluded, padded rows come back as
    zeros and are zeroed again after the output projection, exactly like the
    reference (``torch_transformer_benchmark.py:120-121``).
    """

    def __init__(self, d_model: int, num_heads: int) -> None:
        super().__init__()
        if d_model % num_heads:
            raise ValueError("d_model must be divisible by num_heads")
        self.d_model = d_model
        self.num_heads = num_heads
        self.head_dim = d_model // num_heads
        self.scale = self.head_dim ** -0.5
        self.q_proj = Linear(d_model, d_model)
        self.k_proj = Linear(d_model, d_model)
        self.v_proj = Linear(d_model, d_model)
        self.out_proj = Linear(d_model, d_model)

    def heads_view(self, t: torch.Tensor) -> torch.Tensor:
        """``[B, S, D] -> [B, H, S, dh]`` as a strided view (no copy)."""
        b, s, _ = t.shape
        return t.view(b, s, self.num_heads, self.head_dim).transpose(1, 2)

    def project_qkv(self, x: torch.Tensor):
        return self.heads_view(self.q_proj(x)), self.heads_view(self.k_proj(x)), self.heads_view(self.v_proj(x))

    def folds_biases(self, x: torch.Tensor) -> bool:
        """Whether the q / v projection biases go to the kernel (inference on the GPU)."""
        return (x.is_cuda and not torch.is_grad_enabled() and self.q_proj.bias is not None
                and self.v_proj.bias is not None and self.q_proj.bias.dtype == torch.float32)

    def project_qkv_folded(self, x: torch.Tensor):
        """Bias-free q, k, v head views (fp16 for an fp16 ``x``) and the q / v
        biases the kernel adds (a key bias never changes the attention output)."""
        allowed = x.dtype == torch.float32 and split_products_allowed()
        own = projections(x, (self.q_proj.weight, self.k_proj.weight, self.v_proj.weight), allowed=allowed)
        if own is not None:  # one launch
            return (*map(self.heads_view, own), self.q_proj.bias, self.v_proj.bias)
        return (self.heads_view(project(x, self.q_proj.weight, self.q_proj, "weight", allowed=allowed)),
                self.heads_view(project(x, self.k_proj.weight, self.k_proj, "weight", allowed=allowed)),
                self.heads_view(project(x, self.v_proj.weight, self.v_proj, "weight", allowed=allowed)),
                self.q_proj.bias, self.v_proj.bias)

    def attend(self, q, k, v, valid_len, causal):
        return scaled_dot_product_attention(q, k, v, is_causal=causal, scale=self.scale, valid_len=valid_len)

    def context(self, x, valid_token_mask=None, causal=False, valid_len=None):
        """Attention output before the output projection, ``[B, S, D]`` (a free view)."""
        b, s, _ = x.shape
        if self.folds_biases(x):
            q, k, v, qb, vb = self.project_qkv_folded(x)
            ctx = scaled_dot_product_attention(q, k, v, is_causal=causal, scale=self.scale, valid_len=valid_len,
                                               q_bias=qb, v_bias=vb)
        else:
            q, k, v = self.project_qkv(x)
            ctx = self.attend(q, k, v, valid_len, causal)
        return ctx.transpose(1, 2).reshape(b, s, self.d_model)

    def forward(self, x, valid_token_mask=None, causal=False, valid_len=None):
        out = self.out_proj(self.context(x, valid_token_mask, causal, valid_len))
        if valid_token_mask is not None:
            out = out.masked_fill(~valid_token_mask[..., None], 0)
        return out


class EncoderBlock(nn.Module):
    """Pre-norm residual block with exact GELU (``torch_transformer_benchmark.py:125-145``).

    With ``norm_first=False`` the block is post-norm, ``x = norm1(x +
    attention(x))`` then ``x = norm2(x + ffn(x))``, and ``activation="relu"``
    puts ReLU in the FFN: ``torch.nn.TransformerEncoderLayer``'s semantics for
    those options (dropout off). Same modules and parameter names either way;
    padded rows are zeroed at the end of the block as in the reference.
    """

    def __init__(self, d_model: int, num_heads: int, ffn_dim: int, norm_first: bool = True,
                 activation: str = "gelu") -> None:
        super().__init__()
        if activation not in ACTIVATIONS:
            raise ValueError(f"activation must be one of {ACTIVATIONS}, not {activation!r}")
        self.norm_first = norm_first
        self.activation = activation
        self.norm1 = nn.LayerNorm(d_model)
        self.attention = HipSelfAttention(d_model, num_heads)
        self.norm2 = nn.LayerNorm(d_model)
        self.ffn_in = Linear(d_model, ffn_dim)
        self.ffn_out = Linear(ffn_dim, d_model)

    def _act(self, h: torch.Tensor) -> torch.Tensor:
        return F.gelu(h, approximate="none") if self.activation == "gelu" else F.relu(h)

    def forward(self, x, valid_token_mask, causal, valid_len=None):
        if self._can_fuse(x, valid_token_mask, valid_len):
            return self._forward_fused(x, valid_token_mask, causal, valid_len)
        if self.norm_first:
            x = x + self.attention(self.norm1(x), valid_token_mask, causal, valid_len=valid_len)
            x = x + self.ffn_out(self._act(self.ffn_in(self.norm2(x))))
        else:
            x = self.norm1(x + self.attention(x, valid_token_mask, causal, valid_len=valid_len))
            x = self.norm2(x + self.ffn_out(self._act(self.ffn_in(x))))
        if valid_token_mask is not None:
            x = x.masked_fill(~valid_token_mask[..., None], 0)
        return x

    def _can_fuse(self, x, valid_token_mask, valid_len) -> bool:
        return (x.is_cuda and x.dtype == torch.float32 and x.ndim == 3 and x.is_contiguous()
                and x.data_ptr() % 16 == 0 and x.shape[-1] % 4 == 0 and self.ffn_in.out_features % 4 == 0
                and (valid_token_mask is None or valid_len is not None)
                and self.attention.out_proj.bias is not None and self.ffn_in.bias is not None
                and self.ffn_out.bias is not None
                and (self.norm_first or self._post_norms_fusable(x)))

    def _post_norms_fusable(self, x) -> bool:
        c = x.shape[-1]
        return (c in NORM_WIDTHS
                and all(type(n) is nn.LayerNorm and n.elementwise_affine and n.bias is not None
                        and n.weight.dtype == torch.float32 for n in (self.norm1, self.norm2)))

    def _hidden(self, a, act, allowed):
        """The FFN's fp32 hidden activations, ``act(ffn_in(a))``."""
        own = projections(a, (self.ffn_in.weight,), self.ffn_in.bias, self.activation, allowed)
        if own is not None:
            return own[0]
        return _must(act(_linear_f32(a, self.ffn_in.weight), self.ffn_in.bias))

    def _forward_fused(self, x, valid_token_mask, causal, valid_len):
        """Same computation as the unfused forward; the projection GEMMs run
        bias-free and each bias add, residual add, activation and row zeroing
        is folded into one pass over the GEMM output (for the post-norm block
        together with the LayerNorm that follows it)."""
        if not self.norm_first:
            return self._forward_fused_post(x, valid_token_mask, causal, valid_len)
        from .kernels.elementwise import MODE_ZERO_OUT, MODE_ZERO_Y, bias_gelu, bias_relu, bias_residual

        act = bias_gelu if self.activation == "gelu" else bias_relu
        attn, allowed = self.attention, split_products_allowed()
        ctx = attn.context(self.norm1(x), valid_token_mask, causal, valid_len)
        y = project(ctx, attn.out_proj.weight, attn.out_proj, "weight", allowed=allowed)
        x = _must(bias_residual(x, y, attn.out_proj.bias, valid_len, MODE_ZERO_Y, out=y))
        h = self._hidden(self.norm2(x), act, allowed)
        y = project(h, self.ffn_out.weight, self.ffn_out, "weight", allowed=allowed)
        return _must(bias_residual(x, y, self.ffn_out.bias, valid_len, MODE_ZERO_OUT, out=y))

    def _forward_fused_post(self, x, valid_token_mask, causal, valid_len):
        """The post-norm block: each residual pass stores only the LayerNorm of
        its sum, which is the next residual stream; the second one zeroes the
        padded rows of its norm (the block's final ``masked_fill``)."""
        from .kernels.elementwise import MODE_PLAIN, MODE_ZERO_Y, bias_gelu, bias_relu, bias_residual_layernorm

        act = bias_gelu if self.activation == "gelu" else bias_relu
        attn, allowed = self.attention, split_products_allowed()
        ctx = attn.context(x, valid_token_mask, causal, valid_len)
        y = project(ctx, attn.out_proj.weight, attn.out_proj, "weight", allowed=allowed)
        del ctx
        _, x = _must(bias_residual_layernorm(x, y, attn.out_proj.bias, valid_len, MODE_ZERO_Y, self.norm1,
                                             keep_sum=False))
        del y
        h = self._hidden(x, act, allowed)
        y = project(h, self.ffn_out.weight, self.ffn_out, "weight", allowed=allowed)
        del h
        _, x = _must(bias_residual_layernorm(x, y, self.ffn_out.bias, valid_len, MODE_PLAIN, self.norm2,
                                             zero_padded_norm=valid_token_mask is not None, keep_sum=False))
        return x

    def _forward_fused_norms(self, state, valid_token_mask, causal, valid_len, next_norm, last,
                             fp16_operands=False):
        """``_forward_fused`` that takes ``state = [x, norm1(x)]`` and hands back
        ``(x_out, next_norm(x_out))``: each residual pass also writes the
        LayerNorm its result feeds (``norm2`` here, then the next block's
        ``norm1`` or the final norm, with padded rows zeroed after the last
        block).

        ``state`` is emptied on entry, so this method holds the only
        references to its inputs and every intermediate is released at its
        last use: the largest set alive at once is the residual, the normed
        input, q/k/v and the attention output during attention, and the
        residual, one normed copy and the FFN hidden activation afterwards --
        the working set the streaming planner
        (``implementations.planner``) budgets for.

        ``fp16_operands`` rounds every GEMM input (normed activations, the
        attention output, the GELU output, weights) to fp16 -- the 10-bit
        mantissa of TF32 -- and accumulates in fp32; q, k, v leave their GEMM
        as fp16 (the attention kernel rounds them to fp16 anyway), the other
        GEMM results stay fp32, and so do the residual stream, LayerNorm
        statistics, softmax and GELU. The LayerNorm and GELU kernels write
        their outputs directly as the fp16 operands (no separate cast pass);
        only the final norm, the model's output, stays fp32."""
        from .kernels.elementwise import MODE_ZERO_OUT, MODE_ZERO_Y, bias_gelu, bias_relu, bias_residual_layernorm

        attn, allowed = self.attention, not fp16_operands and split_products_allowed()
        f32, f16 = torch.float32, torch.float16
        x, a = state
        state.clear()
        if fp16_operands and a.dtype != f16:  # the first block's norm1 is a torch LayerNorm
            a = a.half()
        ctx = attn.context(a, valid_token_mask, causal, valid_len)
        del a
        # Layers of width 128: a projection and the passes after it in one.
        own = None if fp16_operands else residual_norm(ctx, attn.out_proj.weight, attn.out_proj.bias, x, valid_len,
                                                       MODE_ZERO_Y, self.norm2, allowed=allowed)
        if own is not None:
            del ctx
            x, a = own
        else:
            y = project(ctx, attn.out_proj.weight, attn.out_proj, "weight", f32, allowed)
            del ctx
            x, a = _must(bias_residual_layernorm(x, y, attn.out_proj.bias, valid_len, MODE_ZERO_Y, self.norm2, out=y,
                                                 norm_dtype=f16 if fp16_operands else f32))
            del y
        own = None if fp16_operands else ffn_norm(a, self.ffn_in.weight, self.ffn_in.bias, self.activation,
                                                  self.ffn_out.weight, self.ffn_out.bias, x, valid_len, MODE_ZERO_OUT,
                                                  next_norm, zero_padded_norm=last and valid_token_mask is not None,
                                                  allowed=allowed)
        if own is not None:
            return own
        act = bias_gelu if self.activation == "gelu" else bias_relu
        if fp16_operands:
            h = project(a, self.ffn_in.weight, self.ffn_in, "weight", f32)
            # the activation straight into the fp16 operand of the next GEMM
            h = _must(act(h, self.ffn_in.bias, out_f16=True))
        else:
            h = self._hidden(a, act, allowed)
        del a
        y = project(h, self.ffn_out.weight, self.ffn_out, "weight", f32, allowed)
        del h
        return _must(bias_residual_layernorm(x, y, self.ffn_out.bias, valid_len, MODE_ZERO_OUT, next_norm, out=y,
                                             zero_padded_norm=last and valid_token_mask is not None,
                                             norm_dtype=f16 if fp16_operands and not last else f32))


def _must(t):
    if t is None:
        raise RuntimeError("the fused block kernels rejected a layout the block checked beforehand")
    return t


class TransformerEncoder(nn.Module):
    """Layer stack plus final LayerNorm (``torch_transformer_benchmark.py:148-172``)."""

    #: "fp32" (default): float32 GEMMs under torch's matmul precision setting.
    #: "fp16": GEMM operands rounded to fp16 with fp32 accumulation (the
    #: mantissa of TF32); fused GPU path only, other paths raise.
    gemm_operands = "fp32"

    def __init__(self, config: TransformerConfig) -> None:
        super().__init__()
        self.config = config
        self.norm_first, self.activation = block_variant(config)
        self.layers = nn.ModuleList(
            EncoderBlock(config.d_model, config.num_heads, config.ffn_dim, self.norm_first, self.activation)
            for _ in range(config.num_layers)
        )
        # A post-norm stack ends in its last block's norm (torch.nn.TransformerEncoder
        # with norm=None); only the pre-norm stack has a final LayerNorm.
        self.final_norm = nn.LayerNorm(config.d_model) if self.norm_first else nn.Identity()

    def forward_layers(self, x, valid_token_mask=None, valid_len=None, gemm_operands=None):
        """The layer stack and final norm; ``gemm_operands`` overrides the
        model's setting for this call."""
        operands = self.gemm_operands if gemm_operands is None else gemm_operands
        if operands not in ("fp32", "fp16"):
            raise ValueError(f"gemm_operands must be 'fp32' or 'fp16', not {operands!r}")
        if self._can_fuse_norms(x, valid_token_mask, valid_len):
            return self._forward_layers_fused(x, valid_token_mask, valid_len, operands)
        if operands == "fp16":
            from .errors import UnsupportedCaseError

            raise UnsupportedCaseError("fp16 GEMM operands are implemented on the fused pre-norm GPU path only")
        for layer in self.layers:
            x = layer(x, valid_token_mask, self.config.causal, valid_len=valid_len)
        if not self.norm_first:
            return x  # each block already ended in its norm and its row zeroing
        x = self.final_norm(x)
        if valid_token_mask is not None:
            x.masked_fill_(~valid_token_mask[..., None], 0)  # x is the norm's fresh output
        return x

    def _can_fuse_norms(self, x, valid_token_mask, valid_len) -> bool:
        d = x.shape[-1] if x.ndim == 3 else 0
        if not self.norm_first:
            return False
        norms = [m for layer in self.layers for m in (layer.norm1, layer.norm2)] + [self.final_norm]
        return (len(self.layers) > 0 and d in NORM_WIDTHS
                and all(layer._can_fuse(x, valid_token_mask, valid_len) for layer in self.layers)
                and all(type(n) is nn.LayerNorm and n.elementwise_affine and n.bias is not None
                        and n.weight.dtype == torch.float32 for n in norms))

    def _forward_layers_fused(self, x, valid_token_mask, valid_len, operands="fp32"):
        """The layer stack with every LayerNorm but the first fused into the
        residual pass before it (same computation as the loop above)."""
        state = [x, self.layers[0].norm1(x)]
        del x
        n = len(self.layers)
        for i, layer in enumerate(self.layers):
            nxt = self.layers[i + 1].norm1 if i + 1 < n else self.final_norm
            state = list(layer._forward_fused_norms(state, valid_token_mask, self.config.causal, valid_len, nxt,
                                                    last=i + 1 == n, fp16_operands=operands == "fp16"))
        return state[1]

    def forward(self, x, valid_token_mask: Optional[torch.Tensor] = None):
        valid_len = None if valid_token_mask is None else prefix_lengths(valid_token_mask)
        return self.forward_layers(x, valid_token_mask, valid_len)


def prefix_lengths(valid_token_mask: torch.Tensor) -> torch.Tensor:
    """Device int32 ``[B]`` valid lengths of a right-padded mask; raises on any other mask.

    One host synchronisation (the prefix check). The dispatcher caches the
    result per mask tensor so timed loops never pay it.
    """
    if valid_token_mask.ndim != 2 or valid_token_mask.dtype != torch.bool:
        raise ValueError("valid_token_mask must be a two-dimensional bool tensor")
    lengths = valid_token_mask.sum(dim=1, dtype=torch.int32)
    pos = torch.arange(valid_token_mask.shape[1], device=valid_token_mask.device)
    if not bool(torch.equal(valid_token_mask, pos[None, :] < lengths[:, None])):
        from .errors import UnsupportedCaseError

        raise UnsupportedCaseError(
            "the HIP attention kernels take right-padded (prefix) masks only; "
            "left padding or interior gaps are not supported"
        )
    return lengths
