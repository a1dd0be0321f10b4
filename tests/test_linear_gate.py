"""When the split-bf16 dense layers may stand in for a float32 product (CPU):
exactly where the product itself would run in hipBLASLt's fast mode."""

from __future__ import annotations

import subprocess
import sys
from pathlib import Path

import pytest
import torch

ROOT = Path(__file__).resolve().parent.parent

# A process of its own: the settings are global and cannot all be set back.
_PROBE = """
import sys, types, torch
from techjam_amd.kernels.linear import _usable
x = types.SimpleNamespace(is_cuda=True, dtype=torch.float32, device=torch.device("cuda", 0),
                          get_device=lambda: 0, is_contiguous=lambda: True, data_ptr=lambda: 0)
mm = torch.backends.cuda.matmul
exec(sys.argv[1])
with torch.no_grad():
    print(bool(_usable(None, x)))
"""


@pytest.mark.parametrize("settings,usable", [
    ("", False),
    ("torch.set_float32_matmul_precision('high')", True),
    ("torch.set_float32_matmul_precision('medium')", True),
    ("mm.allow_tf32 = True", True),
    ("mm.fp32_precision = 'tf32'", True),
    ("torch.backends.fp32_precision = 'tf32'", True),
    ("torch.set_float32_matmul_precision('highest')", False),
    ("torch.set_float32_matmul_precision('high'); mm.fp32_precision = 'ieee'", False),
    ("torch.set_float32_matmul_precision('high'); mm.allow_tf32 = False", False),
    ("torch.set_float32_matmul_precision('high'); torch.backends.cuda.preferred_blas_library('cublas')", False),
    ("torch.set_float32_matmul_precision('high'); torch.set_autocast_enabled('cuda', True)", False),
])
def test_the_setting_the_gemms_obey_decides(settings, usable):
    res = subprocess.run([sys.executable, "-c", _PROBE, settings], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert res.returncode == 0, res.stderr[-2000:]
    assert res.stdout.strip() == str(usable)


@pytest.mark.parametrize("size", [(32,), (1,), (128,), (1, 64)])
def test_a_bias_of_another_size_stays_off_the_kernel(monkeypatch, size):
    """The kernel reads as many bias values as the weight has rows."""
    from techjam_amd.kernels import linear

    monkeypatch.setattr(linear, "_usable", lambda *t: [0] * len(t))
    monkeypatch.setattr(linear._lib, "lib", lambda: pytest.fail("the kernel would be called"))
    x, w = torch.zeros(4, 128), torch.zeros(64, 128)
    assert linear.projections(x, (w,), torch.zeros(size), "gelu") is None


@pytest.mark.parametrize("tokens,taken", [(24575, False), (24576, True), (122880, True), (131072, False)])
def test_tokens_of_the_one_pass_residual(monkeypatch, tokens, taken):
    """At 131 072 tokens and more the library's product and one pass are faster."""
    from techjam_amd.kernels import linear

    asked = []
    monkeypatch.setattr(linear, "_residual_ok", lambda *a: asked.append(a))
    x, w, b = torch.empty(1, tokens, 128, device="meta"), torch.zeros(128, 128), torch.zeros(128)
    assert linear.residual_norm(x, w, b, x, None, 0, torch.nn.LayerNorm(128)) is None
    assert bool(asked) == taken
