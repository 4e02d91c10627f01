"""Which layers past the short-prompt kernel's length still take it: the masks that a coverage can make at most decide, not the sparse
ones of vertical-slash heads alone (CPU: the rule is the host's)."""

import types

import pytest
import torch

from shareprefill_amd import shareprefill_attn


def taken(n, d, pattern, min_budget=1024, opens=False, stride=1):
    sharing = types.SimpleNamespace(opens_cluster=lambda layer, hq: opens, max_pivots=lambda layer, hq: 8)
    k = torch.empty(1).expand(1, 1, n, d).as_strided((1, 1, 1, d), (0, 0, stride * d, 0))
    return shareprefill_attn._short_in_steady_layers(sharing, 1, 32, n, d, pattern, -(-min_budget // 128), k, k)


@pytest.mark.parametrize("d,pattern,last", [(128, 0.65, 11264), (128, 0.9, 7680), (128, 0.95, 6656), (64, 0.65, 131072), (64, 0.95, 131072),
                                            (64, 0.99, 65536), (64, 0.995, 32768)])
def test_a_layer_of_query_aware_heads_is_even_at_the_line(d, pattern, last):
    """Measured there (csrc/sp_attn_short.hip): at 8192 tokens and 0.9 such a layer took 562 us in the short-prompt kernel, 552 in the
    persistent one, at 16384 and 0.65 1201 and 1157."""
    assert taken(last, d, pattern) and not taken(last + 1, d, pattern)
    assert not taken(last, d, pattern, opens=True)


def test_a_minimum_budget_that_makes_masks_dense_keeps_the_persistent_kernel():
    assert taken(8192, 128, 0.65, min_budget=1280) and not taken(8192, 128, 0.65, min_budget=2048)
    assert not taken(7168, 128, 0.9, min_budget=3584)
    assert taken(65536, 64, 0.9, min_budget=32768)  # 64 channels: ahead on any mask


def test_offsets_inside_a_block_have_32_bits():
    assert not taken(8192, 64, 0.9, stride=2 ** 18)
