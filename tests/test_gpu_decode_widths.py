"""The decode step at the head sizes and cache lengths where its instances and its launches change, by the check and the bounds of
test_gpu_decode.py."""

import pytest
from test_gpu_decode import test_decode_batch_matches_oracle as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [8, 40, 64, 72, 120, 128])
@pytest.mark.parametrize("b,hq,hkv,n", [(1, 4, 2, 1), (2, 8, 1, 129), (1, 14, 2, 1100), (1, 40, 4, 700), (2, 17, 1, 300)])
def test_head_sizes(gpu_device, b, hq, hkv, n, d):
    check(gpu_device, b, hq, hkv, n, d)


@pytest.mark.parametrize("b,n", [(1, 128), (1, 255), (1, 256), (2, 257), (1, 383), (1, 384), (2, 385), (16, 257)])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (12, 12, 64), (16, 1, 128), (30, 1, 32)])
def test_caches_of_a_few_tiles(gpu_device, b, n, hq, hkv, d):
    """One workgroup walks the chunks of a cache of up to two tiles; three are three chunks, or fewer in a batch."""
    check(gpu_device, b, hq, hkv, n, d)


@pytest.mark.parametrize("b,n", [(1, 128), (1, 256), (3, 200)])
def test_no_scratch_where_none_is_asked_for(gpu_device, b, n):
    """Where the size function says zero bytes a caller may have allocated nothing: hipMalloc(0) gives a null pointer."""
    import torch

    from shareprefill_amd import _lib, ops

    hq, hkv, d = 8, 2, 128
    lib = _lib.load()
    assert lib.sp_decode_batch_workspace_bytes(b, n, hq, hkv) == 0
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    q, k, v = (torch.randn(b, h, m, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h, m in ((hq, 1), (hkv, n), (hkv, n)))
    want = ops.decode_attention_batch(q, k, v, d ** -0.5)
    out = torch.full_like(want, float("nan"))
    rc = lib.sp_decode_attn_batch_bf16(q.data_ptr(), k.data_ptr(), v.data_ptr(), b, n, hq, hkv, d, q.stride(0), q.stride(1), k.stride(0),
                                       k.stride(2), k.stride(1), v.stride(0), v.stride(2), v.stride(1), d ** -0.5, out.data_ptr(),
                                       None, 0, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "sp_decode_attn_batch_bf16")
    assert torch.equal(out, want)
    n = 257  # one tile more: partials, and a null workspace is refused as ever
    assert lib.sp_decode_batch_workspace_bytes(1, n, hq, hkv) > 0
    k, v = (torch.zeros(1, hkv, n, d, device=gpu_device, dtype=torch.bfloat16) for _ in range(2))
    with pytest.raises(ValueError, match="null workspace"):
        _lib.check(lib.sp_decode_attn_batch_bf16(q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, n, hq, hkv, d, q.stride(0), q.stride(1),
                                                 k.stride(0), k.stride(2), k.stride(1), v.stride(0), v.stride(2), v.stride(1),
                                                 d ** -0.5, out.data_ptr(), None, 0, 0), "sp_decode_attn_batch_bf16")


@pytest.mark.parametrize("d", [8, 64, 72, 128])
@pytest.mark.parametrize("hq,hkv", [(6, 2), (34, 2)])  # the ring kernel's splits, whose padded widths leave part of a partial; the other kernel's
def test_scratch_may_hold_anything(gpu_device, hq, hkv, d):
    """The second kernel takes nothing from the scratch that the first has not written."""
    import torch

    from shareprefill_amd import _lib, ops

    b, n = 2, 4000
    gen = torch.Generator(device=gpu_device).manual_seed(d)
    q, k, v = (torch.randn(b, h, m, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h, m in ((hq, 1), (hkv, n), (hkv, n)))
    need = _lib.load().sp_decode_batch_workspace_bytes(b, n, hq, hkv)
    assert need > 0
    outs = []
    for byte in (0, 0xFF):  # (zeros, NaN)
        scratch = ops._workspace("decode", need, gpu_device)
        scratch.fill_(byte)
        outs.append(ops.decode_attention_batch(q, k, v, d ** -0.5))
        assert (scratch != byte).any(), "this call leaves no partials: it does not test what it is for"
    assert outs[0].isfinite().all() and torch.equal(outs[0], outs[1])
