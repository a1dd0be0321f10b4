"""The polynomial kernel's split of a sixteen-chunk window into parts (GPU).

Fewer than 16 heads fold each window in two parts (a part starts from the
window's start plus the first part's sum), 16 or more in one. Lengths around
the ends of parts and windows: a window of 16 chunks is 8192 tokens, a part
4096.
"""

from __future__ import annotations

import pytest
import torch

from oracle.poly import coefficient_table, poly_linear_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [1, 15, 16])
@pytest.mark.parametrize("n", [512, 513, 4097, 4608, 4609, 8192, 8705, 12801, 16896, 25089])
def test_windows_and_parts_match_the_oracle_scan(cuda, n, heads):
    from techjam_amd.kernels.poly import poly_rows

    g = torch.Generator(device=cuda).manual_seed(n + heads)
    q, k, v = (torch.randn(1, n, heads, 64, generator=g, device=cuda).transpose(1, 2) * s for s in (0.5, 0.5, 1.0))
    scale = 64 ** -0.5
    coeffs = coefficient_table(torch.full((1, heads), 0.25))
    got = poly_rows(q, k, v, scale, coeffs.float().reshape(-1, 3).to(cuda), exact_prefix=0)
    torch.cuda.synchronize()
    # The first and the last head: the others run the same code on other data.
    for h in {0, heads - 1}:
        sl = slice(h, h + 1)
        ref = poly_linear_attention(q[:, sl].cpu(), k[:, sl].cpu(), v[:, sl].cpu(), scale, chunk=512, exact_prefix=0,
                                    coeffs=coeffs[:, sl])
        out = got[:, sl].cpu()
        rel = float((out.double() - ref.double()).norm() / ref.double().norm())
        # fp16 operands and state shadows: each product off by at most about
        # 3 * 2^-11, random in sign; a part that is lost or counted twice
        # shows as an error of order one.
        assert rel < 3 * 2 ** -11, (h, rel)
        assert bool(torch.isfinite(out).all())
