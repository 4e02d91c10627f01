"""shareprefill_attention_forward runs the core under its module's name, also one that a caller put there."""

import types

import pytest
import torch

from shareprefill_amd import shareprefill_attn as sa


@pytest.mark.parametrize("n", [2, 700])
def test_a_callers_core_is_called(monkeypatch, n):
    seen = []

    def core(module, q, k, v, gqa_interleave=False):
        seen.append(gqa_interleave)
        return q + 1, None

    monkeypatch.setattr(sa, "shareprefill_attention_core", core)
    q = torch.randn(1, 4, n, 8)
    out, _ = sa.shareprefill_attention_forward(types.SimpleNamespace(), q, q, q, None, scaling=1.0, gqa_interleave=True)
    assert seen == [True] and out.is_contiguous()
    torch.testing.assert_close(out, (q + 1).transpose(1, 2), rtol=0, atol=0)
