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


def test_width_128_ffn_with_relu(cuda):
    from techjam_amd.kernels.linear import ffn_norm

    b, s = 2, 12301
    x, r, w, w2, bi, bo, *g = _draw(cuda, 5, (b, s, 128), (b, s, 128), (128, 128), (128, 128), (128,), (128,), (128,),
                                    (128,))
    norm, xs = _norm(cuda, g), x.reshape(-1, 128)
    h = F.relu(xs.double() @ w.double().t() + bi.double())
    hidden = _bound(xs, w) + 1e-6 * (1 + h)
    bound = (hidden @ w2.double().abs().t() + _bound(h + hidden, w2)).view(b, s, 128)
    ref = r.double() + (h @ w2.double().t() + bo.double()).view(b, s, 128)
    _check_residual(ffn_norm(x, w, bi, "relu", w2, bo, r, None, 0, norm), ref, bound, norm)


@pytest.mark.parametrize("tokens", [1, 31, 4100])
def test_sum_in_place_or_not_stored(cuda, tokens):
    """The two forms of ``out`` that only the C entry points offer: the
    residual itself, and none."""
    from techjam_amd.kernels import _lib
    from techjam_amd.kernels.attention import _stream_ptr

    x, r, w, w2, bi, bo, ga, be = _draw(cuda, tokens, (tokens, 128), (tokens, 128), (128, 128), (128, 128), (128,),
                                        (128,), (128,), (128,))
    lib, stream = _lib.lib(), _stream_ptr(x.device)

    def residual(resid, out, ln):
        return lib.tj_narrow_residual_norm(x.data_ptr(), w.data_ptr(), bo.data_ptr(), resid.data_ptr(), out, tokens, tokens,
                                           None, 0, ga.data_ptr(), be.data_ptr(), ln.data_ptr(), 1e-5, 0, stream)

    def ffn(resid, out, ln):
        return lib.tj_narrow_ffn_norm(x.data_ptr(), w.data_ptr(), bi.data_ptr(), 2, w2.data_ptr(), bo.data_ptr(),
                                      resid.data_ptr(), out, tokens, tokens, None, 0, ga.data_ptr(), be.data_ptr(),
                                      ln.data_ptr(), 1e-5, 0, stream)

    for call in (residual, ffn):
        out, ln = torch.empty_like(r), torch.empty_like(r)
        assert call(r, out.data_ptr(), ln) == 0
        inplace, ln_in = r.clone(), torch.empty_like(r)
        assert call(inplace, inplace.data_ptr(), ln_in) == 0
        ln_only = torch.empty_like(r)
        assert call(r, None, ln_only) == 0
        torch.cuda.synchronize()
        assert torch.equal(inplace, out) and torch.equal(ln_in, ln) and torch.equal(ln_only, ln)
        assert bool(torch.isfinite(ln).all())


@pytest.mark.parametrize("m,n,k,n_w", [(256, 256, 256, 1), (96, 128, 512, 3), (30000, 128, 128, 1), (30000, 128, 128, 3)])
def test_infinities_nan_and_huge_values(cuda, m, n, k, n_w):
    """An infinite or NaN input, or one past bf16's largest, makes its row NaN
    (the low part of an infinity is inf - inf), as in the library's fast mode;
    the other rows do not see it."""
    from techjam_amd.kernels.linear import projections

    x, *ws = _draw(cuda, n + k, (m, k), *[(n, k)] * n_w)
    rows = [3, 7, 11, 20, m - 1]
    for row, value in zip(rows, (float("inf"), float("nan"), 3.4e38, -float("inf"), -3.4e38)):
        x[row, row % k] = value
    clean = torch.ones(m, dtype=torch.bool, device=cuda)
    clean[rows] = False
    for w, y in zip(ws, projections(x, ws)):
        assert bool(torch.isnan(y[rows]).all())
        assert bool(torch.equal(torch.isnan(y), torch.isnan(F.linear(x, w))))
        assert bool(((y[clean].double() - x[clean].double() @ w.double().t()).abs() <= _bound(x[clean], w)).all())


def test_a_nan_token_stays_in_its_row_of_a_width_128_block(cuda):
    from techjam_amd.kernels.linear import ffn_norm, residual_norm

    b, s = 1, 24576
    x, r, w, w2, bi, bo, *g = _draw(cuda, 9, (b, s, 128), (b, s, 128), (128, 128), (128, 128), (128,), (128,), (128,),
                                    (128,))
    norm = _norm(cuda, g)
    lengths = torch.tensor([s - 10], dtype=torch.int32, device=cuda)
    clean = [t.clone() for t in (*residual_norm(x, w, bo, r, lengths, 2, norm),
                                 *ffn_norm(x, w, bi, "gelu", w2, bo, r, lengths, 2, norm))]
    x[0, 100, 5], x[0, s - 1, 7] = float("nan"), float("inf")  # a valid row and a padded one
    got = (*residual_norm(x, w, bo, r, lengths, 2, norm), *ffn_norm(x, w, bi, "gelu", w2, bo, r, lengths, 2, norm))
    for was, now in zip(clean, got):
        assert bool(torch.isnan(now[0, 100]).all())
        now[0, 100] = was[0, 100]
        assert torch.equal(now, was)  # the padded row is zeroed, not multiplied by zero
