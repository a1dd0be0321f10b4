"""fp32 heads of 256, and of 128 with split scores, run on 32-key tiles: lengths
around the ends of a key tile and of a query tile, against brute force (GPU)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.attention import brute_force_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,split", [(256, False), (128, True)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("s", [1, 31, 32, 33, 64, 65, 127, 129, 289])
def test_thirty_two_key_tiles(cuda, s, causal, d, split):
    from techjam_amd.kernels import scaled_dot_product_attention

    g = torch.Generator().manual_seed(1000 * d + s)
    q, k, v = (torch.randn(2, s, 3, d, generator=g).transpose(1, 2) for _ in range(3))
    lengths = torch.tensor([s, max(1, s - 17)], dtype=torch.int32)
    got = scaled_dot_product_attention(q.to(cuda), k.to(cuda), v.to(cuda), is_causal=causal, qk_split=split,
                                       valid_len=lengths.to(cuda))
    torch.cuda.synchronize()
    ref = np.asarray(brute_force_attention(q, k, v, d ** -0.5, causal, valid_len=lengths.tolist()), dtype=np.float64)
    got = got.double().cpu().numpy()
    for i, n in enumerate(lengths.tolist()):
        # v rounded to fp16 (half an ulp, 2^-11 of sum p |v| <= 2^-11 max |v|);
        # without split scores q, k and P too: scores off by at most 2^-10 of
        # sum |q k| scale, which moves an output by twice that times max |v|.
        vmax = float(v[i].abs().max())
        bound = 2 ** -11 * vmax + 1e-5
        if not split:
            qk = float((q[i].double().abs() @ k[i].double().abs().transpose(-2, -1)).max()) * d ** -0.5
            bound += vmax * (2 ** -11 + 2 * 2 ** -10 * qk)
        assert np.abs(got[i, :, :n] - ref[i, :, :n]).max() <= bound
        assert not got[i, :, n:].any()
