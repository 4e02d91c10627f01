"""The decode step's ring kernel where its cuts change: slices of one, two, four and eight channel tiles, splits of the keys, last steps
of every kind, against the attention in 64 bits.  The output is rounded to bf16 once (at most 2^-9 of a value each, so of the 2-norm);
everything before that -- products of bf16 values in fp32, probabilities as two bf16 values, 2^-17 -- is held to 2 % of that."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 1.02 * 2.0 ** -9


def _exact(q, k, v, scale):
    b, hq, _, d = q.shape
    hkv = k.shape[1]
    q, k, v = (t.double() for t in (q, k, v))
    p = torch.softmax(torch.matmul(q.reshape(b, hkv, hq // hkv, d), k.transpose(2, 3).contiguous()) * scale, -1)
    return torch.matmul(p, v).reshape(b, 1, hq, d)


def _error(out, want):
    return ((out.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("b,hq,hkv,n,d", [
    (1, 4, 2, 33, 128), (1, 32, 8, 257, 128), (1, 32, 8, 1025, 128), (3, 28, 4, 700, 128),  # one tile of channels: eight waves
    (8, 32, 8, 225, 128), (5, 128, 8, 449, 128), (12, 32, 8, 193, 128), (11, 9, 9, 385, 128),  # two and four: seven, six
    (33, 8, 8, 129, 128), (3, 24, 8, 5000, 128),  # all of them in a slice, without and with splits
    (5, 16, 8, 300, 64), (13, 16, 8, 289, 64), (40, 16, 8, 100, 64), (2, 14, 2, 9001, 64),
    (1, 6, 2, 1025, 96), (9, 8, 8, 300, 40), (2, 16, 1, 4000, 72)])
@pytest.mark.parametrize("token_major", [False, True])
def test_against_64_bits(gpu_device, b, hq, hkv, n, d, token_major):
    from shareprefill_amd import ops

    gen = torch.Generator(device=gpu_device).manual_seed(b * n + d)
    mk = lambda *s: torch.randn(*s, generator=gen, device=gpu_device).to(torch.bfloat16)
    q = mk(b, hq, 1, d)
    if token_major:  # rows wider than the head, with NaN behind it
        wide = lambda: torch.nn.functional.pad(mk(b, n, hkv, d), (0, 8), value=float("nan"))[..., :d].transpose(1, 2)
        k, v = wide(), wide()
    else:
        k, v = mk(b, hkv, n, d), mk(b, hkv, n, d)
    k[:, :, n // 2] *= 3
    out = ops.decode_attention_batch(q, k, v, d ** -0.5)
    assert _error(out, _exact(q, k, v, d ** -0.5)) <= BOUND
    assert torch.equal(out, ops.decode_attention_batch(q, k, v, d ** -0.5))


@pytest.mark.parametrize("hq,hkv", [(8, 2), (24, 2)])  # that kernel's instances of up to 8 and 16 heads a group
@pytest.mark.parametrize("n,d", [(200, 128), (1025, 64), (3000, 96)])
def test_results_on_odd_addresses_and_caches_of_one_row_a_token(gpu_device, n, d, hq, hkv):
    """A result that no wide store may write, and keys that are one row for every token (a stride of zero): the former goes to the
    other kernel, whose probabilities are one bf16 value (2^-8 more)."""
    from shareprefill_amd import _lib, ops

    gen = torch.Generator(device=gpu_device).manual_seed(n)
    mk = lambda *s: torch.randn(*s, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(1, hq, 1, d), mk(1, hkv, n, d), mk(1, hkv, n, d)
    want = _exact(q, k, v, d ** -0.5)
    room = torch.empty(hq * d + 1, dtype=torch.bfloat16, device=gpu_device)
    lib = _lib.load()
    ws = torch.empty(max(1, lib.sp_decode_batch_workspace_bytes(1, n, hq, hkv)), dtype=torch.uint8, device=gpu_device)
    rc = lib.sp_decode_attn_batch_bf16(q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, n, hq, hkv, d, 0, q.stride(1), 0, k.stride(2), k.stride(1),
                                       0, v.stride(2), v.stride(1), d ** -0.5, room.data_ptr() + 2, ws.data_ptr(), ws.numel(),
                                       torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "sp_decode_attn_batch_bf16")
    assert _error(room[1:].view(1, 1, hq, d), want) <= 2.0 ** -8
    one = k[:, :, :1].expand(1, hkv, n, d)
    assert one.stride(2) == 0
    out = ops.decode_attention_batch(q, one, v, d ** -0.5)
    assert _error(out, _exact(q, one, v, d ** -0.5)) <= BOUND


@pytest.mark.parametrize("b,n", [(1, 300), (1, 3000)])  # one launch; splits
def test_keys_whose_logits_are_minus_infinity(gpu_device, b, n):
    """Keys that no query can see, among them whole steps, whole waves' shares and a whole split: they weigh nothing."""
    from shareprefill_amd import ops

    hq, hkv, d = 8, 2, 128
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    mk = lambda *s: torch.randn(*s, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(b, hq, 1, d).abs(), mk(b, hkv, n, d), mk(b, hkv, n, d)
    seen = torch.ones(n, dtype=torch.bool, device=gpu_device)
    seen[:70] = seen[128:256] = seen[260:290:2] = False
    k[:, :, ~seen] = k[:, :, ~seen].abs()
    k[:, :, ~seen, 5] = float("-inf")
    want = _exact(q, k[:, :, seen], v[:, :, seen], d ** -0.5)
    assert _error(ops.decode_attention_batch(q, k, v, d ** -0.5), want) <= BOUND


@pytest.mark.parametrize("b,hq,hkv,n,d", [(1, 8, 2, 300, 128), (1, 8, 2, 3000, 128), (12, 32, 8, 193, 128), (33, 8, 8, 129, 128),
                                          (1, 14, 2, 1025, 64), (1, 6, 2, 1025, 96), (80, 16, 8, 100, 128)])  # slices of every width, splits
def test_values_that_are_infinite(gpu_device, b, hq, hkv, n, d):
    """A channel whose values hold one infinity is that infinity, and NaN where they hold both, as in 64 bits: the probabilities'
    second part is zero for some keys and negative for others.  The other channels do not notice."""
    from shareprefill_amd import ops

    gen = torch.Generator(device=gpu_device).manual_seed(n)
    mk = lambda *s: torch.randn(*s, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(b, hq, 1, d), mk(b, hkv, n, d), mk(b, hkv, n, d)
    keys = torch.randperm(n - 1, generator=gen, device=gpu_device)[:d]  # (the last key also stands in for those behind the cache, weight 0)
    channels = torch.arange(0, d, 2, device=gpu_device)  # one infinity in every other channel, the second sign in some
    sign = 1.0 - 2.0 * (channels % 4 == 0)
    v[:, :, keys[:d // 2], channels] = (sign * float("inf")).to(torch.bfloat16)
    v[:, :, keys[d // 2:d // 2 + 3], channels[:3]] = (-sign[:3] * float("inf")).to(torch.bfloat16)
    q[0, 0] = 0  # equal weights, all of them bf16 values: no second part
    out, want = ops.decode_attention_batch(q, k, v, d ** -0.5), _exact(q, k, v, d ** -0.5)
    assert torch.equal(out.isnan(), want.isnan()) and want[..., channels[:3]].isnan().all()
    inf = want.isinf()
    assert inf[..., channels[3:]].all() and torch.equal(out[inf].double(), want[inf])
    rest = want.isfinite()
    assert _error(out[rest], want[rest]) <= BOUND


@pytest.mark.parametrize("hq,hkv", [(40, 2), (17, 1), (32, 1)])  # the kernel of groups of 17 to 32 heads
@pytest.mark.parametrize("b,n,d", [(1, 256, 128), (300, 512, 128), (1, 3000, 128), (1, 3000, 64)])  # two chunks and four of a workgroup; splits
def test_keys_whose_logits_are_minus_infinity_in_large_groups(gpu_device, b, n, d, hq, hkv):
    """The other kernel's case of test_keys_whose_logits_are_minus_infinity: whole tiles of 128 keys, which are chunks and splits of
    their own, have no key that a query can see.  Probabilities are one bf16 value there (2^-8 more)."""
    from shareprefill_amd import ops

    gen = torch.Generator(device=gpu_device).manual_seed(n)
    mk = lambda *s: torch.randn(*s, generator=gen, device=gpu_device).to(torch.bfloat16)
    q, k, v = mk(b, hq, 1, d).abs(), mk(b, hkv, n, d), mk(b, hkv, n, d)
    seen = torch.ones(n, dtype=torch.bool, device=gpu_device)
    seen[:128] = seen[256:384] = seen[140:170:2] = seen[2816:] = False
    k[:, :, ~seen] = k[:, :, ~seen].abs()
    k[:, :, ~seen, 5] = float("-inf")
    out = ops.decode_attention_batch(q, k, v, d ** -0.5)
    some = sorted({0, b // 2, b - 1})
    assert _error(out[some], _exact(q[some], k[some][:, :, seen], v[some][:, :, seen], d ** -0.5)) <= BOUND + 2.0 ** -8


@pytest.mark.parametrize("b,hq,hkv,n,d", [
    (33, 16, 8, 97, 128), (64, 16, 8, 501, 128), (300, 2, 1, 1, 128), (33, 24, 8, 300, 64), (512, 1, 1, 31, 64),  # two workgroups a CU
    (65, 16, 8, 33, 128), (65, 8, 8, 400, 128), (200, 28, 4, 64, 128), (513, 1, 1, 1, 128), (65, 16, 8, 800, 64), (520, 7, 1, 65, 64),  # four
    (65, 8, 8, 533, 96), (65, 16, 8, 711, 72),  # four, rows as long as they are
    (65, 8, 8, 401, 128), (65, 8, 8, 801, 64), (65, 8, 8, 534, 96),  # one
    (40, 8, 8, 300, 96), (65, 16, 8, 257, 72), (40, 8, 8, 300, 40), (70, 16, 8, 129, 8)])
def test_more_pairs_of_sequence_and_kv_head_than_cus(gpu_device, b, hq, hkv, n, d):
    test_against_64_bits(gpu_device, b, hq, hkv, n, d, False)
    test_against_64_bits(gpu_device, b, hq, hkv, n, d, True)
