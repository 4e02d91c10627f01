"""64-channel heads run unpadded on short prompts, whose kernels read 16 bytes at a time: inputs whose storage does not
allow that are copied, not refused."""

import types

import pytest
import torch

from shareprefill_amd import shareprefill_attn


def odd_offset(t):
    """t's values, contiguous, at a storage offset of one element."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    view = buf[1:].view(t.shape)
    view.copy_(t)
    return view


def odd_head_stride(t):
    """t [1, 1, N, D] with a head stride that means nothing but is odd."""
    return t.as_strided(t.shape, (t.stride(0), 7, t.stride(2), t.stride(3)))


def channel_strided(t):
    return t.repeat_interleave(2, dim=3)[..., ::2]


def odd_token_stride(t):
    return torch.nn.functional.pad(t, (0, 3))[..., :t.shape[3]]


VIEWS = [odd_offset, odd_head_stride, channel_strided, odd_token_stride]


@pytest.mark.parametrize("view", VIEWS)
def test_unreadable_rows_are_copied(view):
    t = torch.randn(1, 1, 5, 64).to(torch.bfloat16)
    v = view(t)
    assert torch.equal(v, t)
    got = shareprefill_attn._rows_16_byte_aligned(v)
    assert torch.equal(got, t)
    assert got.data_ptr() % 16 == 0 and got.stride(3) == 1 and all(s % 8 == 0 for s in got.stride()[:-1])
    assert shareprefill_attn._rows_16_byte_aligned(got) is got


def test_token_strides_beyond_32_bit_offsets_are_copied():
    t = torch.zeros(1, 1, 1, 64, dtype=torch.bfloat16)
    for stride, copied in ((2 ** 24 - 8, False), (2 ** 24, True)):  # (one token: nothing is read through the stride)
        far = t.as_strided((1, 1, 1, 64), (64, 64, stride, 1))
        assert (shareprefill_attn._rows_16_byte_aligned(far) is not far) == copied


@pytest.mark.gpu
@pytest.mark.parametrize("n", [700, 1500])  # all blocks kept; selected
@pytest.mark.parametrize("view", VIEWS)
def test_views_give_the_same_bits(gpu_device, tmp_path, n, view):
    from shareprefill_amd import AttentionSharing, synthetic

    path = synthetic.write_cluster_table(synthetic.random_cluster_table(4, 1, 1, 3), str(tmp_path / "table.json"))
    cfg = types.SimpleNamespace(block_size=128, min_budget=1024, max_budget=None, pattern_threshold=0.9, similarity_threshold=0.5,
                                fallback_threshold=0.9, queryaware_threshold=0.1)
    q, k, v = synthetic.planted_qkv(4, 1, n, 64, 1, device=gpu_device, q_head_gain=1.0)

    def run(*qkv):
        mod = types.SimpleNamespace(config=cfg, attention_sharing=AttentionSharing(path), layer_idx=0, scaling=0.125)
        return shareprefill_attn.shareprefill_attention_core(mod, *qkv)

    want = run(*(t.contiguous() for t in (q, k, v)))
    got = run(q if view is odd_head_stride else view(q), view(k.contiguous()), view(v.contiguous()))
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
