"""The split-bf16 dense layers against float64 on the GPU.

Element by element: a product of split operands misses lo.lo (at most 2^-16 of
|x||w|) and the rounding of both lo parts (2^-17 each), and the fp32 sums add
K * 2^-24, so an output is within (2^-14 + K * 2^-24) * sum |x||w| of the
exact one.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def fast_float32():
    prev = torch.get_float32_matmul_precision()
    torch.set_float32_matmul_precision("high")
    with torch.no_grad():
        yield
    torch.set_float32_matmul_precision(prev)


def _draw(cuda, seed, *shapes):
    g = torch.Generator(device=cuda).manual_seed(seed)
    return [torch.randn(*s, generator=g, device=cuda) for s in shapes]


def _bound(x, w):
    k = w.shape[1]
    return (2 ** -14 + k * 2 ** -24) * (x.double().abs() @ w.double().abs().t())


@pytest.mark.parametrize("m,n,k,n_w", [(1, 32, 64, 1), (31, 96, 192, 2), (33, 256, 256, 3), (64, 64, 512, 1),
                                       (130, 128, 448, 3), (1, 128, 128, 3), (2000, 128, 128, 3), (4099, 128, 128, 2)])
def test_projections(cuda, m, n, k, n_w):
    from techjam_amd.kernels.linear import projections

    x, *ws = _draw(cuda, m + n + k, (m, k), *[(n, k)] * n_w)
    got = projections(x, ws)
    for w, y in zip(ws, got):
        assert bool(((y.double() - x.double() @ w.double().t()).abs() <= _bound(x, w)).all())


@pytest.mark.parametrize("m", [21760, 21761, 21889, 65536])
def test_three_projections_over_the_whole_chip(cuda, m):
    """One turn of the resident workgroups (170 per weight, 128 tokens each), and more."""
    from techjam_amd.kernels.linear import projections

    x, *ws = _draw(cuda, m, (m, 128), *[(128, 128)] * 3)
    for w, y in zip(ws, projections(x, ws)):
        assert bool(((y.double() - x.double() @ w.double().t()).abs() <= _bound(x, w)).all())


@pytest.mark.parametrize("act", ["gelu", "relu"])
@pytest.mark.parametrize("m,n,k", [(7, 128, 64), (65, 1024, 256), (40, 32, 512)])
def test_hidden_layer(cuda, m, n, k, act):
    from techjam_amd.kernels.linear import projections

    x, w, b = _draw(cuda, m, (m, k), (n, k), (n,))
    y, = projections(x, (w,), b, act)
    pre = x.double() @ w.double().t() + b.double()
    ref = F.gelu(pre) if act == "gelu" else F.relu(pre)
    # both activations have slopes below 1.13; fp32 erf and products on top
    assert bool(((y.double() - ref).abs() <= 1.13 * _bound(x, w) + 1e-6 * (1 + pre.abs())).all())


def _norm(cuda, g):
    norm = torch.nn.LayerNorm(128, device=cuda)
    norm.weight.copy_(1 + 0.1 * g[0])
    norm.bias.copy_(0.1 * g[1])
    return norm


def _check_residual(got, ref_out, bound, norm):
    out, ln = got
    assert bool(((out.double() - ref_out).abs() <= bound + 1e-6 * (1 + ref_out.abs())).all())
    # LayerNorm of the stored sum: fp32 statistics of 128 values
    ref_ln = F.layer_norm(out.double(), (128,), norm.weight.double(), norm.bias.double(), norm.eps)
    assert bool(((ln.double() - ref_ln).abs() <= 1e-5 * (1 + ref_ln.abs())).all())


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("b,s", [(3, 8201), (192, 128)])
def test_width_128_passes(cuda, b, s, mode):
    from techjam_amd.kernels.linear import ffn_norm, residual_norm

    x, r, w, w2, bi, bo, *g = _draw(cuda, b, (b, s, 128), (b, s, 128), (128, 128), (128, 128), (128,), (128,), (128,),
                                    (128,))
    norm = _norm(cuda, g)
    lengths = torch.tensor([s if i == 0 else (37 * i) % s for i in range(b)], dtype=torch.int32, device=cuda)
    ok = (torch.arange(s, device=cuda)[None] < lengths[:, None])[..., None]
    xs, rs = x.reshape(-1, 128), r.double()

    def combine(y):
        y = y.view(b, s, 128)
        return rs + y if mode == 0 else (torch.where(ok, rs + y, 0 * y) if mode == 2 else rs + torch.where(ok, y, 0 * y))

    y = xs.double() @ w.double().t() + bo.double()
    bound = _bound(xs, w).view(b, s, 128)
    _check_residual(residual_norm(x, w, bo, r, lengths, mode, norm), combine(y), bound, norm)

    pre = xs.double() @ w.double().t() + bi.double()
    h = F.gelu(pre)
    y = h @ w2.double().t() + bo.double()
    # the hidden error (slope below 1.13) through |w2|, and the second product's own
    hidden = 1.13 * _bound(xs, w) + 1e-6 * (1 + pre.abs())
    bound = (hidden @ w2.double().abs().t() + _bound(h.abs() + hidden, w2)).view(b, s, 128)
    _check_residual(ffn_norm(x, w, bi, "gelu", w2, bo, r, lengths, mode, norm), combine(y), bound, norm)
    zeroed = ffn_norm(x, w, bi, "gelu", w2, bo, r, lengths, mode, norm, zero_padded_norm=True)[1]
    assert torch.count_nonzero(zeroed.masked_select(~ok)).item() == 0


def test_refusals_leave_the_library_to_it(cuda):
    from techjam_amd.kernels.linear import projections

    x, w = _draw(cuda, 0, (64, 128), (64, 128))
    assert projections(x.t().contiguous().t(), (w,)) is None  # not row-major
    assert projections(x[:, :100].contiguous(), (w[:, :100].contiguous(),)) is None  # K not a multiple of 64
    assert projections(x.double(), (w.double(),)) is None
    with torch.enable_grad():
        assert projections(x, (w,)) is None
    torch.set_float32_matmul_precision("highest")
    assert projections(x, (w,)) is None


def test_autocast_decides_the_type_of_the_attention_context(cuda):
    from techjam_amd.model import HipSelfAttention

    x, = _draw(cuda, 1, (2, 64, 256))
    attn = HipSelfAttention(256, 4).to(cuda).eval()
    with torch.autocast("cuda", torch.float16):
        assert attn.context(x).dtype == torch.float16
    assert attn.context(x).dtype == torch.float32
