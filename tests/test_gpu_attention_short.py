"""GPU parity of the short-prompt attention kernel with the fp32 masked-attention oracle (bounds and their derivation:
test_gpu_attention.py; the block-average maps add the probabilities as rounded to bf16, 2^-9 relative each, and are compared
to 2^-8)."""

import numpy as np
import pytest
import torch

from oracle import shareprefill_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_REL = 2e-2, 2.5e-3


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,n", [(8, 8, 1), (8, 1, 65), (16, 4, 130), (4, 2, 640), (7, 1, 1111),
                                      (32, 8, 2048),   # the last size whose rows are split over two sets of waves
                                      (32, 8, 2177),   # the first that is not; ragged by one token
                                      (3, 1, 8300)])   # more than one mask word per row
def test_short_attention_matches_oracle(gpu_device, hq, hkv, n, d):
    """Random masks with dense heads among them, whose maps the kernel writes; logits that grow along the row for the last
    head, so that the running max has to move past its headroom."""
    from shareprefill_amd import ops

    gen = torch.Generator().manual_seed(n + d)
    mk = lambda h: torch.randn(n, h, d, generator=gen).to(torch.bfloat16).transpose(0, 1)
    q, k, v = mk(hq), mk(hkv), mk(hkv)
    k[-1] *= (1 + 9 * torch.arange(n) / n)[:, None].to(torch.bfloat16)
    nb = -(-n // 128)
    rng = np.random.default_rng(n)
    mask = np.tril(rng.random((hq, nb, nb)) < 0.4)
    mask[:, np.arange(nb), np.arange(nb)] = True
    mask[:, :, 0] = True
    dense = np.arange(hq) % 3 == 1
    mask[dense] = np.tril(np.ones((nb, nb), dtype=bool))
    decision = torch.where(torch.from_numpy(dense), O.DEC_DENSE, O.DEC_VS).to(torch.int32)
    ref, maps = O.masked_attention(q, k, v, mask, 128, d ** -0.5, want_avg=dense)
    avg = torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device)
    bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
    qg, kg, vg = q.to(gpu_device), k.to(gpu_device), v.to(gpu_device)
    out = ops.short_attention(qg, kg, vg, bits, d ** -0.5, decision.to(gpu_device), avg)
    assert out.shape == (n, hq, d)
    cleared = torch.full_like(avg, 7.0)
    plain = ops.short_attention(qg, kg, vg, bits, d ** -0.5, avg_attn=cleared)
    assert torch.equal(out, plain)  # (a head's output does not depend on whether its map is wanted)
    assert not cleared.any()
    out, ref = out.transpose(0, 1).float().cpu(), ref.float()
    assert (out - ref).abs().max().item() <= MAX_ABS
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL
    avg = avg.cpu().numpy()
    assert not avg[~dense].any()
    for h in np.nonzero(dense)[0]:
        assert np.abs(avg[h] - np.asarray(maps[h])).max() <= 2.0 ** -8
