"""sp_select_layer_repack_bf16: the key-major copy of V made beside the selection is the one sp_attn_repack_v_bf16 makes, bit for
bit, and the selection is that of sp_select_layer_bf16."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,n,bs,transposed", [
    (2, 1, 1025, 128, False),    # nine tiles, the last of one token
    (7, 1, 2048, 128, True),     # whole tiles, head-major strides
    (4, 4, 300, 64, False),      # a smaller block size: the tiles stay 128 keys wide
    (3, 3, 6657, 128, True),
    (2, 2, 131200, 128, False),  # beyond the lengths whose budgets are part of the launch
])
def test_repack_beside_the_selection(gpu_device, hq, hkv, n, bs, transposed):
    from shareprefill_amd import _lib, ops

    gen = torch.Generator(device=gpu_device).manual_seed(n)

    def mk(h):
        t = torch.randn((h, n, 128) if transposed else (n, h, 128), generator=gen, device=gpu_device).to(torch.bfloat16)
        return t if transposed else t.transpose(0, 1)

    q, k, v = mk(hq), mk(hkv), mk(hkv)
    nb = -(-n // bs)
    hc = torch.full((hq,), -1, dtype=torch.int32, device=gpu_device)
    tiles = hkv * -(-n // 128) * 128 * 128 * 2
    want, got = (torch.full((tiles,), 0xA5, dtype=torch.uint8, device=gpu_device) for _ in range(2))
    ops.repack_v(v, bs, want)
    res = []
    for repack in (None, (v, got)):
        probs = torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device)
        mask, ints, _ = ops.select_layer(ops.ClusterState(0, nb, gpu_device), hc, 0, q, k, bs, _lib.SP_FLAG_LOGITS_BF16, 8, nb, 0.9,
                                         0.5, 0.9, 0.1, probs, repack=repack)
        res.append((mask, ints))
    assert torch.equal(want, got)
    assert torch.equal(res[0][0], res[1][0])
    assert all(torch.equal(a, b) for a, b in zip(res[0][1], res[1][1]))
    with pytest.raises(RuntimeError):  # a buffer one byte short
        ops.select_layer(ops.ClusterState(0, nb, gpu_device), hc, 0, q, k, bs, _lib.SP_FLAG_LOGITS_BF16, 8, nb, 0.9, 0.5, 0.9, 0.1,
                         probs, repack=(v, got[:-1]))
    with pytest.raises(ValueError):
        ops.select_layer(ops.ClusterState(0, nb, gpu_device), hc, 0, q, k, bs, _lib.SP_FLAG_LOGITS_BF16, 8, nb, 0.9, 0.5, 0.9, 0.1,
                         probs, repack=(v[:, 1:], got))
