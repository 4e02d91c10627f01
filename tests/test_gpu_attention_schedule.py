"""The work distribution of the persistent attention kernel (slots, pairing, ranking of the gangs) at the sizes where it can
go wrong, through what depends on it: every (row, head) must be computed exactly once and pivots must find their slots.
Bounds and their derivation: test_gpu_attention.py (outputs), test_gpu_attention_short.py (maps)."""

import numpy as np
import pytest
import torch

from oracle import shareprefill_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_REL = 2e-2, 2.5e-3


@pytest.mark.parametrize("hq,hkv,n,max_pivots", [
    (3, 1, 8193, 1),     # ranked; an odd head count, an odd block count, the last block one token; more pivots than slots
    (4, 4, 8320, 8),     # no two heads share a kv head: nothing may be paired by heads
    (66, 2, 8200, 70),   # more heads than a wave, more gangs than one round of half-waves, groups of 33
    (6, 2, 8192, 0),     # one block below the ranked range
    (5, 5, 32896, 2),    # one block above it
])
def test_every_row_once_and_pivots_in_their_slots(gpu_device, hq, hkv, n, max_pivots):
    from shareprefill_amd import _lib, ops

    d = 128
    gen = torch.Generator().manual_seed(n)
    mk = lambda h: torch.randn(n, h, d, generator=gen).to(torch.bfloat16).transpose(0, 1)
    q, k, v = mk(hq), mk(hkv), mk(hkv)
    nb = -(-n // 128)
    rng = np.random.default_rng(n)
    mask = np.tril(rng.random((hq, nb, nb)) < 3.0 / nb)
    mask[:, np.arange(nb), np.arange(nb)] = True
    mask[1::2] = mask[0::2][: len(mask[1::2])]  # adjacent heads keep the same blocks: pairing by heads is the better one
    pivot = np.arange(hq) % 3 == 2
    decision = torch.where(torch.from_numpy(pivot), O.DEC_DENSE, O.DEC_VS).to(torch.int32)
    heads = np.arange(hq) if hq <= 6 else np.array([h for h in (0, 1, 2, 31, 32, 33, 64, 65, 127, 128, 200, 254, 255) if h < hq])
    group = hq // hkv
    kv = torch.from_numpy(heads // group)
    ref, maps = O.masked_attention(q[heads], k[kv], v[kv], mask[heads], 128, d ** -0.5, want_avg=pivot[heads])
    avg = torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device)
    bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
    assert _lib.load().sp_short_attn_max_tokens(d) < n
    args = (q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), bits, 128, d ** -0.5)
    kw = dict(decision=decision.to(gpu_device), max_pivots=max_pivots, workspace=ops.attention_workspace(
        n, hq, hkv, d, 128, gpu_device, max_pivots))
    ops.repack_v(args[2], 128, kw["workspace"][0])
    # NaN stands where the output goes (the allocator hands the block that was just freed out again), so that a row of any head
    # that nothing writes is seen
    poison = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    where = poison.data_ptr()
    del poison
    out = ops.block_sparse_attention(*args, avg_attn=avg, **kw)
    assert out.data_ptr() == where
    assert torch.isfinite(out).all()
    out, ref = out.transpose(0, 1)[heads].float().cpu(), ref.float()
    assert (out - ref).abs().max().item() <= MAX_ABS
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL
    avg = avg.cpu().numpy()
    assert not avg[~pivot].any()
    for i, h in enumerate(heads):
        if pivot[h]:
            assert np.abs(avg[h] - np.asarray(maps[i])).max() <= 2.0 ** -8
    by_heads = ops.attention_pairing(n, hq, hkv, d, 128, gpu_device)
    slots = min(max_pivots, int(pivot.sum()))
    slotted = set(np.nonzero(pivot)[0][:slots].tolist())
    for i, yes in enumerate(by_heads):
        h0, h1 = 2 * i, 2 * i + 1
        may = h1 < hq and h0 // group == h1 // group and not ({h0, h1} & slotted)
        assert bool(yes) == bool(may)  # (equal masks: the union by heads is the smaller one wherever it is allowed)
