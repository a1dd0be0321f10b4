"""Few query tiles with long key sweeps: the sweep is cut into parts that a
second kernel adds (GPU). Against the one-sweep kernel of the same library --
which the exact-attention tests hold to the oracle -- and against float64
softmax attention."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _one_sweep(q, k, v, causal, lengths, q_bias, v_bias):
    """The same call without a workspace."""
    from techjam_amd.kernels import _lib
    from techjam_amd.kernels.attention import _DTYPES, _stream_ptr, empty_like_heads

    out = empty_like_heads(q)
    b, h, s, d = q.shape
    code = _lib.lib().tj_attn_fwd_proj_bias(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), _DTYPES[q.dtype], b, h, s, d,
        *(_lib.strides4(t) for t in (q, k, v, out)), d ** -0.5, int(causal),
        None if lengths is None else lengths.data_ptr(), None if q_bias is None else q_bias.data_ptr(),
        None if v_bias is None else v_bias.data_ptr(), _stream_ptr(q.device))
    assert code == 0
    return out


# Around the ends of parts (multiples of 512 keys and of 128 rows), one to
# many parts a tile, several (b, h) per XCD and fewer than eight.
@pytest.mark.parametrize("b,h,s,d,dtype", [
    (1, 1, 1281, 64, torch.float32), (1, 2, 2048, 64, torch.float16), (2, 3, 2049, 64, torch.float32),
    (1, 1, 5000, 32, torch.float16), (1, 4, 3583, 128, torch.float32), (1, 1, 2177, 128, torch.float16),
    (1, 2, 2500, 256, torch.float32), (1, 9, 4096, 64, torch.float16), (1, 1, 1537, 256, torch.float16), (1, 1, 2176, 64, torch.float32),
    (1, 1, 16384, 64, torch.float32), (2, 2, 2049, 64, torch.float32)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("padded,biased", [(False, False), (True, True)])
def test_parts_add_up(cuda, b, h, s, d, dtype, causal, padded, biased):
    from techjam_amd.kernels import _lib, scaled_dot_product_attention

    if _lib.lib().tj_attn_workspace_bytes(b, h, s, d, int(causal)) == 0:
        pytest.skip("one part")
    g = torch.Generator(device=cuda).manual_seed(s + d)
    q, k, v = (torch.randn(b, s, h, d, generator=g, device=cuda).to(dtype).transpose(1, 2) for _ in range(3))
    # lengths that leave whole parts, and whole tiles, without keys
    lengths = torch.tensor([s // 3 + 1] + [0] * (b - 1), dtype=torch.int32, device=cuda) if padded else None
    qb, vb = ((torch.randn(h * d, generator=g, device=cuda) for _ in range(2)) if biased else (None, None))
    got = scaled_dot_product_attention(q, k, v, is_causal=causal, valid_len=lengths, q_bias=qb, v_bias=vb)
    want = _one_sweep(q, k, v, causal, lengths, qb, vb)
    torch.cuda.synchronize()
    # The same fp16 scores and products; references differ between parts, so P
    # is rounded at other points: 2^-11 of sum p |v| / l each way.
    vmax = float((v if vb is None else v + vb.view(1, h, 1, d)).abs().max())
    tol = 2 * 2 ** -11 * vmax + (2 ** -10 * vmax if dtype == torch.float16 else 1e-5)
    assert float((got.float() - want.float()).abs().max()) <= tol
    n = s if lengths is None else int(lengths[0])
    assert lengths is None or torch.count_nonzero(got[0, :, n:]).item() == 0
    # and float64 attention of the first (b, h), at its last rows
    rows = slice(max(0, n - 300), n)
    qd = q[0, 0, rows].double() + (0 if qb is None else qb[:d].double())
    sc = qd @ k[0, 0, :n].double().t() * d ** -0.5
    if causal:
        sc = sc.masked_fill(torch.arange(n, device=cuda)[None] > torch.arange(rows.start, n, device=cuda)[:, None],
                            float("-inf"))
    ref = torch.softmax(sc, -1) @ v[0, 0, :n].double() + (0 if vb is None else vb[:d].double())
    rel = float((got[0, 0, rows].double() - ref).norm() / ref.norm())
    assert rel < 2e-3, rel  # fp16 operands: about 3.5e-4, 4 to 5 times that at the largest


@pytest.mark.parametrize("d,dtype", [(32, torch.float32), (64, torch.float16), (64, torch.float32), (128, torch.float32),
                                     (128, torch.float16)])
def test_split_scores_in_parts(cuda, d, dtype):
    """Flagged and plain heads of one launch, each against the same call on one sweep."""
    from techjam_amd.kernels import _lib, scaled_dot_product_attention
    from techjam_amd.kernels.attention import _DTYPES, _stream_ptr, empty_like_heads

    b, h, s = 1, 3, 2500
    assert _lib.lib().tj_attn_workspace_bytes(b, h, s, d, 1) > 0
    g = torch.Generator(device=cuda).manual_seed(d)
    q, k, v = (torch.randn(b, s, h, d, generator=g, device=cuda).to(dtype).transpose(1, 2) for _ in range(3))
    flags = torch.tensor([1, 0, 1], dtype=torch.int32, device=cuda)
    got = scaled_dot_product_attention(q, k, v, is_causal=True, qk_split=flags)
    want = empty_like_heads(q)
    code = _lib.lib().tj_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), want.data_ptr(), _DTYPES[dtype], b, h, s, d,
                                  *(_lib.strides4(t) for t in (q, k, v, want)), d ** -0.5, 1, None, None,
                                  flags.data_ptr(), _stream_ptr(q.device))
    assert code == 0
    torch.cuda.synchronize()
    vmax = float(v.abs().max())
    tol = torch.tensor([1e-5, 2 * 2 ** -11 * vmax, 1e-5], device=cuda).view(1, 3, 1, 1)  # split heads: only v is rounded
    if dtype == torch.float16:
        tol = tol + 2 ** -10 * vmax  # outputs rounded to fp16 on both sides
    assert bool(((got.float() - want.float()).abs() <= tol).all())


def test_capture_replays_with_the_parts(cuda):
    from techjam_amd.kernels import scaled_dot_product_attention

    # Inference mode throughout: a capture earlier in the process leaves its
    # random state as an inference tensor.
    with torch.inference_mode():
        g = torch.Generator(device=cuda).manual_seed(5)
        q, k, v = (torch.randn(1, 4096, 2, 64, generator=g, device=cuda).transpose(1, 2) for _ in range(3))
        want = scaled_dot_product_attention(q, k, v, is_causal=True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = scaled_dot_product_attention(q, k, v, is_causal=True)
        for _ in range(3):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
            torch.randn(1 << 20, device=cuda).sum().item()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_nan_and_infinite_keys_as_in_one_sweep(cuda, causal, dtype):
    """A row that sees a NaN score is NaN whatever its other parts hold; keys
    that all score -inf weigh nothing, also where a part starts on them."""
    from techjam_amd.kernels import _lib, scaled_dot_product_attention

    b, h, s, d = 1, 2, 4096, 64
    assert _lib.lib().tj_attn_workspace_bytes(b, h, s, d, int(causal)) > 0
    g = torch.Generator(device=cuda).manual_seed(11)
    q, k, v = (torch.randn(b, s, h, d, generator=g, device=cuda).to(dtype).transpose(1, 2) for _ in range(3))
    q[0, 1, :, 0] = q[0, 1, :, 0].abs() + 0.5
    k[0, 0, 2000, 3] = float("nan")
    for t0 in range(512, s, 512):  # whole key tiles at every possible start of a part
        k[0, 1, t0:t0 + 64, 0] = -float("inf")
    got = scaled_dot_product_attention(q, k, v, is_causal=causal)
    want = _one_sweep(q, k, v, causal, None, None, None)
    torch.cuda.synchronize()
    bad = torch.isnan(want).any(-1)
    assert bool(bad[0, 0, -1]) and not bool(bad[0, 1].any())
    assert torch.equal(torch.isnan(got).any(-1), bad)
    tol = 2 * 2 ** -11 * float(v.abs().max()) + (2 ** -10 * float(v.abs().max()) if dtype == torch.float16 else 1e-5)
    assert float((got - want)[~bad].abs().max()) <= tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("level", [-40.0, -200.0, 3.0])
@pytest.mark.parametrize("dead", [64, 192])
def test_low_scores_behind_infinite_keys(cuda, dtype, level, dead):
    """A part that starts on keys scoring -inf weighs its others by their own
    max: against 2^0, scores around 2^-40 would all round to zero."""
    from techjam_amd.kernels import _lib, scaled_dot_product_attention

    b, h, s, d = 1, 2, 4096, 64
    assert _lib.lib().tj_attn_workspace_bytes(b, h, s, d, 1) > 0
    g = torch.Generator(device=cuda).manual_seed(13)
    q, k, v = (torch.randn(b, s, h, d, generator=g, device=cuda).to(dtype).transpose(1, 2) for _ in range(3))
    q[..., 0] = 16.0
    k[..., 0] = level / 2.885390  # 16 k_0 / 8 log2(e): all scores around 2^level, the same rounding in all
    for t0 in range(512, s, 512):
        k[:, :, t0:t0 + dead, 0] = -float("inf")
    got = scaled_dot_product_attention(q, k, v, is_causal=True)
    seen = torch.ones(s, s, dtype=torch.bool, device=cuda).tril() & ~torch.isinf(k[0, 0, :, 0])[None]
    kd = torch.where(torch.isinf(k[0]), 0, k[0]).double()
    sc = (q[0].double() @ kd.transpose(1, 2).contiguous()) * d ** -0.5
    ref = torch.softmax(sc.masked_fill(~seen, float("-inf")), -1) @ v[0].double()
    # P and v rounded to fp16 (2^-11 of max |v| each), scores off by 2^-10 of
    # the spread of the other dims (below 1.5) and 2^-22 of |level|, fp16 results.
    tol = float(v.abs().max()) * (2 * 2 ** -11 + 2 * (1.5 * 2 ** -10 + 2 ** -22 * abs(level)) + 2 ** -11)
    assert float((got[0].double() - ref).abs().max()) <= tol
