"""The guard's sampled-score sums at the edges of its tiles (GPU): samples
that end inside a 32-row block, fewer rows than one block, head dims that end
inside an eight-dim piece, both input types and strided views."""

from __future__ import annotations

import pytest
import torch

from oracle.poly import estimate_sigma_per_head, sample_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("b,h,n,d", [(1, 1, 1, 64), (2, 3, 33, 64), (1, 2, 65, 4), (1, 3, 500, 36), (2, 2, 600, 68),
                                     (1, 2, 2000, 128)])
def test_moments_match_the_oracle(cuda, b, h, n, d, dtype):
    from techjam_amd.kernels import score_guard

    g = torch.Generator().manual_seed(100 * n + d)
    q, k = (torch.randn(b, n, h, d, generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    scale = d ** -0.5
    res = score_guard(q.to(cuda), k.to(cuda), scale, exact_prefix=100)
    torch.cuda.synchronize()
    idx = sample_rows(n, 512, 0)
    s = (q[:, :, idx].double() @ k[:, :, idx].double().transpose(-2, -1)) * scale
    smax = s.abs().amax(dim=(-1, -2)).flatten()
    # fp32 products and sums of d terms: each score within (d + 2) * 2^-24 of
    # sum |q_i k_i| scale, which (d + 2) * 2^-24 * |q| |k| scale bounds.
    bound = float((d + 2) * 2 ** -24 * scale * q.double().norm(dim=-1).max() * k.double().norm(dim=-1).max())
    assert float((res.smax.cpu().double() - smax).abs().max()) <= bound + 2 ** -24 * float(smax.max())
    mean = s.mean(dim=(-1, -2)).flatten()
    # plus the fp32 sums of 16 scores a lane forms before adding in fp64
    assert float((res.mean.cpu().double() - mean).abs().max()) <= bound + 17 * 2 ** -24 * float(smax.max())
    if n > 1:
        ref = estimate_sigma_per_head(q.float(), k.float(), scale, index=idx).flatten()
        assert torch.allclose(res.sigma.cpu().double(), ref, rtol=1e-4, atol=1e-6)
    else:
        assert res.flags.cpu().tolist() == [0] * (b * h)  # one score has no spread


def test_more_heads_than_one_launch_holds(cuda):
    """2^22 workgroups of 1024 threads exceed a launch: the sums run in slices."""
    from techjam_amd.kernels import score_guard

    h, n, d = (1 << 22) + 5, 2, 4
    g = torch.Generator(device=cuda).manual_seed(1)
    q, k = (torch.randn(1, h, n, d, generator=g, device=cuda, dtype=torch.float16) for _ in range(2))
    res = score_guard(q, k, 0.5, ceiling=0.4)
    torch.cuda.synchronize()
    s = (q[0].float() @ k[0].float().transpose(-2, -1).contiguous()).double() * 0.5  # exact products, four-term sums
    assert torch.allclose(res.mean.double(), s.mean(dim=(-1, -2)), rtol=0, atol=1e-6)
    sd = s.flatten(1).std(dim=1)
    # fp32 squares of scores up to 20, cancelling against the mean's
    assert float((res.sigma.double() - sd).abs().max()) <= 2e-3
    clear = (sd - 0.4).abs() > 2e-3
    assert torch.equal((res.flags == 1)[clear], (sd <= 0.4)[clear])
