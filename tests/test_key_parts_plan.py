"""What the callers of the exact kernel take for granted about its key parts
(CPU: the library's own sizes)."""

from __future__ import annotations

import pytest

from techjam_amd.implementations import planner
from techjam_amd.kernels import _lib


def _bytes(b, h, s, d, causal=1):
    return int(_lib.lib().tj_attn_workspace_bytes(b, h, s, d, causal))


@pytest.mark.parametrize("h,s,d", [(1, 16384, 64), (4, 4096, 128), (2, 5184, 256), (64, 16384, 64), (16, 128, 64)])
def test_the_plan_counts_the_sums_of_key_parts(h, s, d):
    out = h * s * d * 4
    sums = max(_bytes(1, h, s, d, causal) for causal in (0, 1))
    assert planner.attention_core_bytes(1, h, s, d, poly=False) == out + sums
    assert (sums > 0) == (h * s <= 16384 and s > 1216)


@pytest.mark.parametrize("d", [32, 64, 128, 256])
def test_the_sums_fit_the_allowance(d):
    sizes = [*range(1216, 60000, 320), *range(60000, 600000, 8192)]
    most = max(_bytes(1, h, s, d, c) for h in (1, 2, 3, 5, 8, 13, 32, 64, 128) for s in sizes for c in (0, 1))
    assert 0 < most <= 47 << 20 < planner.LIBRARY_ALLOWANCE_BYTES // 4


def test_short_calls_need_not_ask():
    """The largest sequence that no shape cuts into parts, exactly."""
    from techjam_amd.kernels.attention import ONE_SWEEP_MAX_SEQ, SUPPORTED_HEAD_DIMS

    shapes = [(h, d, c) for h in (1, 2, 4, 8, 16, 64) for d in SUPPORTED_HEAD_DIMS for c in (0, 1)]
    assert not any(_bytes(1, h, s, d, c) for h, d, c in shapes for s in range(1, ONE_SWEEP_MAX_SEQ + 1))
    assert any(_bytes(1, h, ONE_SWEEP_MAX_SEQ + 1, d, c) for h, d, c in shapes)


@pytest.mark.parametrize("h,s,d,causal,parts", [
    (1, 2048, 64, 1, True), (1, 16384, 64, 1, True), (8, 2048, 64, 1, True), (4, 4096, 128, 1, True), (4, 1257, 64, 1, True),
    # 2.5 parts' length and more, but the sums of that many parts cost what they save
    (16, 1375, 64, 0, False), (8, 2863, 64, 0, False), (12, 2014, 128, 0, False), (108, 1256, 32, 1, False),
    (6, 1600, 256, 0, True),  # not at head_dim 256
    # less than 2.5
    (16, 4096, 64, 1, False), (32, 2048, 64, 1, False),
])
def test_where_parts_pay(h, s, d, causal, parts):
    assert (_bytes(1, h, s, d, causal) > 0) == parts
