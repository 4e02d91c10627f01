"""What the attention kernels lose against the attention in 64 bits, on inputs where the bound can be derived.

The probabilities enter P.V as bf16, relative to the running maximum.  Where every one of them is a bf16 value relative to
the row's largest, nothing is rounded there, and the output may be off by its own rounding to bf16 (half a unit in the
last place) and by fp32 arithmetic (below 2^-16) only; the pivots' maps, which stay fp32, by the latter alone."""

import pytest
import torch

from shareprefill_amd import _lib, ops

pytestmark = pytest.mark.gpu

LN2 = 0.6931471805599453  # softmax scale under which logits are in octaves
FP32 = 2.0 ** -16         # a few hundred fp32 operations of 2^-24, and the hardware's exp2 / log2


def logit_keys(logits, d):
    """k [len, d] bf16 and the logits in 64 bits that q = (1, 1, 1, 0, ...) gets from them: each in three bf16 parts."""
    k = torch.zeros(len(logits), d, dtype=torch.bfloat16)
    rest = logits.double()
    for c in range(3):
        k[:, c] = rest.to(torch.bfloat16)
        rest = rest - k[:, c].double()
    return k, k.double().sum(1)


def half_ulp(x):
    """of bf16 values of x's size: 8 significant bits"""
    return torch.ldexp(torch.ones_like(x), torch.frexp(x)[1] - 9)


def bf16_weights(n, seed):
    """n values of (1/2, 1] that bf16 holds, the first 1."""
    gen = torch.Generator().manual_seed(seed)
    w = torch.randint(128, 256, (n,), generator=gen) / 256.0
    w[0] = 1.0
    return w


# kernel: 0 = the persistent one, else head_dim of the short-prompt one
@pytest.mark.parametrize("kernel,hq,hkv", [(0, 2, 1), (128, 2, 1), (64, 2, 1), (128, 136, 17), (64, 136, 17)])
@pytest.mark.parametrize("seed", [0, 1])
def test_weights_that_bf16_holds_are_not_rounded(gpu_device, kernel, hq, hkv, seed):
    """The first block's logits lie some octaves, and a fraction of one, below 32 keys of the second block that decide the
    row; the running maximum has to go to their largest, or all of them are rounded at another fraction."""
    n, d = 512, kernel or 128
    w = bf16_weights(32, seed)
    logits = torch.full((n,), -60.0)
    logits[:128] = -9.37
    logits[128:160] = 1.2345 + torch.log2(w)
    k1, exact_logits = logit_keys(logits, d)
    p = torch.softmax(exact_logits * LN2, 0)
    q = torch.zeros(hq, n, d, dtype=torch.bfloat16)
    q[:, :, :3] = 1.0
    v1 = torch.zeros(n, d, dtype=torch.bfloat16)
    v1[128:160, :32] = torch.eye(32)
    k, v = (t.expand(hkv, n, d).contiguous().to(gpu_device) for t in (k1, v1))
    q = q.to(gpu_device)
    mask = ops.bool_to_mask(torch.ones(4, 4, dtype=torch.bool).tril().expand(hq, 4, 4)).to(gpu_device)
    decision = torch.full((hq,), _lib.SP_DEC_DENSE, dtype=torch.int32, device=gpu_device)
    avg = torch.zeros(hq, 4, 4, dtype=torch.float32, device=gpu_device)
    if kernel == 0:
        out = ops.block_sparse_attention(q, k, v, mask, 128, LN2, decision, avg, max_pivots=hq)
    else:
        out = ops.short_attention(q, k, v, mask, LN2, decision, avg)
    got = out[384:, :, :32].double().cpu()  # the last block's queries see all 512 keys but the masked ones of their own block
    want = p[128:160]
    excess = ((got - want).abs() - half_ulp(want)) / want
    assert excess.max().item() <= FP32
    blocks = p.view(4, 128).sum(1)[:2]
    assert ((avg[:, 3, :2].double().cpu() - blocks).abs() / blocks).max().item() <= FP32
