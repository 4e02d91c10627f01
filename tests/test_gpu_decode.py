"""GPU parity of the decode step (one query token per head against the whole KV cache) with the fp32 oracle.

Tolerance: max-abs <= 2e-2, mean-rel <= 2.5e-3 -- the output is rounded to bf16 (unit roundoff 2^-8 -> 1.3e-3
mean-rel on its own); the kernel itself works in fp32 on the bf16 inputs."""

import math

import pytest
import torch

from oracle import shareprefill_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_REL = 2e-2, 2.5e-3


def _inputs(hq, hkv, n, seed, token_major=True, d=128):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(hq, d, generator=g).to(torch.bfloat16)
    if token_major:  # the layout of a Hugging Face cache after transpose: [N, Hkv, D] storage viewed as [Hkv, N, D]
        k = torch.randn(n, hkv, d, generator=g).to(torch.bfloat16).transpose(0, 1)
        v = torch.randn(n, hkv, d, generator=g).to(torch.bfloat16).transpose(0, 1)
    else:
        k = torch.randn(hkv, n, d, generator=g).to(torch.bfloat16)
        v = torch.randn(hkv, n, d, generator=g).to(torch.bfloat16)
    return q, k, v


@pytest.mark.parametrize("hq,hkv,n", [(32, 8, 4096), (28, 4, 1000), (8, 8, 129), (4, 1, 1), (16, 2, 70000),
                                      (8, 1, 127), (18, 2, 3000), (64, 4, 2500), (24, 1, 777), (64, 2, 4096)])
@pytest.mark.parametrize("token_major", [True, False])
def test_decode_matches_oracle(gpu_device, hq, hkv, n, token_major):
    from shareprefill_amd import ops

    q, k, v = _inputs(hq, hkv, n, n + hq, token_major)
    scale = 1.0 / math.sqrt(128)
    ref = O.decode_attention(q, k, v, scale)
    out = ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), scale).cpu().float()
    assert (out - ref).abs().max().item() <= MAX_ABS
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL
    again = ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), scale).cpu().float()
    assert torch.equal(out, again)


@pytest.mark.parametrize("d", [64, 32, 16, 8, 96])
@pytest.mark.parametrize("token_major", [True, False])
def test_decode_smaller_heads_read_the_cache_as_it_is(gpu_device, d, token_major):
    """head_dim below 128 (the reference's 16 / 32 / 64, shareprefill_attn.py:503-508, and any other multiple of 8):
    the kernel pads the rows inside LDS, the cache is neither copied nor padded.  The result must also equal, bit for
    bit, the head_dim-128 call on explicitly zero-padded tensors."""
    from shareprefill_amd import ops

    hq, hkv, n = 12, 4, 3001
    q, k, v = _inputs(hq, hkv, n, 40 + d, token_major, d)
    scale = 1.0 / math.sqrt(d)
    ref = O.decode_attention(q, k, v, scale)
    out = ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), scale)
    assert out.shape == (hq, d)
    o = out.cpu().float()
    assert (o - ref).abs().max().item() <= MAX_ABS
    assert ((o - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL
    pad = lambda t: torch.nn.functional.pad(t, (0, 128 - d)).to(gpu_device)
    wide = ops.decode_attention(pad(q), pad(k), pad(v), scale)
    assert torch.equal(wide[:, :d], out) and float(wide[:, d:].abs().max()) == 0.0


def test_decode_peaked_and_large_logits(gpu_device):
    """A key that dominates (logit far above the rest) and large-magnitude logits: the online softmax across
    tiles and chunks must neither overflow nor lose the winner."""
    from shareprefill_amd import ops

    q, k, v = _inputs(8, 2, 5000, 3)
    k = k.clone()
    k[:, 3333] = (q.float().view(2, 4, 128).mean(1) * 4).to(torch.bfloat16)  # strongly aligned with the queries
    scale = 1.0
    ref = O.decode_attention(q, k, v, scale)
    out = ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), scale).cpu().float()
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max().item() <= 4e-2  # values of magnitude up to ~4: bf16 ulp 0.03
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL


def test_decode_rejects_unsupported(gpu_device):
    from shareprefill_amd import ops

    q, k, v = _inputs(33, 1, 256, 1)
    with pytest.raises(NotImplementedError):
        ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), 0.1)  # 33 heads per kv head
    q, k, v = _inputs(4, 2, 256, 1)
    qg = torch.zeros(4, 132, dtype=torch.bfloat16, device=gpu_device)[:, 4:]  # rows start 8 bytes off a 16-byte line
    qg.copy_(q)
    with pytest.raises(NotImplementedError):
        ops.decode_attention(qg, k.to(gpu_device), v.to(gpu_device), 0.1)
    q, k, v = _inputs(4, 2, 256, 1)
    with pytest.raises(ValueError):
        ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), 0.0)
    for d in (136, 256):  # wider than the kernel's tiles
        q, k, v = _inputs(4, 2, 256, 1, d=d)
        with pytest.raises(NotImplementedError):
            ops.decode_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), 0.1)


@pytest.mark.parametrize("b,hq,hkv,n,d", [(1, 8, 2, 1, 128), (3, 8, 2, 127, 128), (5, 28, 4, 129, 128), (2, 14, 2, 2049, 64),
                                          (64, 8, 8, 300, 128), (65, 16, 8, 128, 64)])
def test_decode_batch_matches_oracle(gpu_device, b, hq, hkv, n, d):
    """Every sequence of a batch against the fp32 oracle: one key, ragged tiles, caches cut into several chunks and
    caches that are a single chunk each (enough sequences to fill the chip: the kernel writes the result itself)."""
    from shareprefill_amd import ops

    gen = torch.Generator().manual_seed(b * n)
    mk = lambda h, m: torch.randn(b, h, m, d, generator=gen).to(torch.bfloat16)
    q, k, v = mk(hq, 1), mk(hkv, n), mk(hkv, n)
    scale = d ** -0.5
    out = ops.decode_attention_batch(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), scale).cpu().float()
    assert out.shape == (b, 1, hq, d)
    for i in sorted({0, b // 2, b - 1}):
        ref = O.decode_attention(q[i, :, 0], k[i], v[i], scale)
        assert (out[i, 0] - ref).abs().max().item() <= MAX_ABS
        assert ((out[i, 0] - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL


# Groups of 17 to 32 heads: the four tiles of a cache are a workgroup each, two to a workgroup, all in one.  Smaller groups: splits, one
# launch of a workgroup to a CU, more than CUs.
@pytest.mark.parametrize("b", [1, 128, 600])
@pytest.mark.parametrize("hq,hkv", [(40, 2), (4, 2)])
@pytest.mark.parametrize("d", [64, 128])
def test_decode_weights_that_bf16_holds_are_not_rounded(gpu_device, b, hq, hkv, d):
    """The probabilities of a chunk are rounded to bf16 relative to the chunk's largest, whatever the other sequences of
    the batch (groups of 17 heads and more; those of smaller groups are two bf16 values): keys whose weights in their tile are bf16
    values keep them, though the tiles' largest logits lie fractions of an octave apart."""
    from shareprefill_amd import ops
    from tests.test_gpu_attention_precision import FP32, LN2, bf16_weights, half_ulp, logit_keys

    n = 512
    logits = torch.full((n,), -60.0)
    for tile, top in enumerate((3.3, 2.55, 1.9, 2.87)):
        logits[128 * tile:128 * tile + 16] = top + torch.log2(bf16_weights(16, tile))
    k1, exact_logits = logit_keys(logits, d)
    p = torch.softmax(exact_logits * LN2, 0)
    q = torch.zeros(b, hq, 1, d, dtype=torch.bfloat16)
    q[..., :3] = 1.0
    v1 = torch.zeros(n, d, dtype=torch.bfloat16)
    for tile in range(4):  # channel 16 tile + i: the weight of the tile's key i
        v1[128 * tile:128 * tile + 16, 16 * tile:16 * tile + 16] = torch.eye(16)
    k, v = (t.expand(b, hkv, n, d).contiguous().to(gpu_device) for t in (k1, v1))
    out = ops.decode_attention_batch(q.to(gpu_device), k, v, LN2)[..., :64].double().cpu()
    want = p.view(4, 128)[:, :16].reshape(64)
    assert (((out - want).abs() - half_ulp(want)) / want).max().item() <= FP32


@pytest.mark.parametrize("b", [65535, 65536, 131075])
def test_decode_batches_past_the_grid_limit(gpu_device, b):
    """A grid's last axis ends at 65535: larger batches go in several launches, every sequence with its own queries and
    cache.  With one key per sequence the output is that key's value."""
    from shareprefill_amd import ops

    gen = torch.Generator(device=gpu_device).manual_seed(b)
    mk = lambda h: torch.randn(b, h, 1, 8, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(2), mk(1), mk(1)
    out = ops.decode_attention_batch(q, k, v, 0.3)
    assert torch.equal(out, v.expand(b, 2, 1, 8).transpose(1, 2))
    # two keys: the first and the last sequence against the oracle
    k, v = mk(2).view(b, 1, 2, 8), mk(2).view(b, 1, 2, 8)
    out = ops.decode_attention_batch(q, k, v, 0.3)
    for i in (0, 65534, b - 1):
        ref = O.decode_attention(q[i, :, 0].cpu(), k[i].cpu(), v[i].cpu(), 0.3)
        assert (out[i, 0].cpu().float() - ref).abs().max().item() <= MAX_ABS


def test_decode_reads_a_larger_cache_up_to_the_batch(gpu_device):
    """A cache kept for more sequences than the step has (and v for more than k)."""
    from shareprefill_amd import ops

    gen = torch.Generator(device=gpu_device).manual_seed(1)
    mk = lambda b, h, m: torch.randn(b, h, m, 64, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(2, 4, 1), mk(3, 2, 300), mk(5, 2, 300)
    assert torch.equal(ops.decode_attention_batch(q, k, v, 0.125), ops.decode_attention_batch(q, k[:2], v[:2], 0.125))
    for bad in ((q, k[:1], v), (q, k, v[:1]), (q, k, v[:, :, :299])):
        with pytest.raises(ValueError):
            ops.decode_attention_batch(*bad, 0.125)


def test_decode_reads_k_and_v_up_to_what_the_step_needs(gpu_device):
    """k says how many heads and tokens there are, q how many channels: v may hold more of all three and k more channels;
    a k or v that holds less is refused."""
    from shareprefill_amd import ops

    gen = torch.Generator(device=gpu_device).manual_seed(2)
    mk = lambda h, m, d: torch.randn(2, h, m, d, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(4, 1, 64), mk(2, 300, 128), mk(3, 417, 96)
    got = ops.decode_attention_batch(q, k, v, 0.125)
    assert torch.equal(got, ops.decode_attention_batch(q, k[..., :64], v[:, :2, :300, :64], 0.125))
    for b in range(2):
        assert torch.equal(ops.decode_attention_batch(q[b:b + 1], k[b:b + 1], v[b:b + 1], 0.125)[0, 0],
                           ops.decode_attention(q[b, :, 0], k[b], v[b], 0.125))
    for bad in ((q, k[..., :56], v), (q, k, v[..., :56]), (q, k, v[:, :1]), (q, k, v[:, :, :299])):
        with pytest.raises(ValueError):
            ops.decode_attention_batch(*bad, 0.125)
