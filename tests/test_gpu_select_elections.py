"""Decisions made by every workgroup of the mask launch for itself (up to 128 blocks) against the election's own launch: some heads
of a cluster query-aware, clusters with a pivot but no pattern yet, slots that do not exist, the most heads."""

import pytest
import torch

from shareprefill_amd import AttentionSharing, _lib, ops, synthetic
from test_gpu_select_layer import _stages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,n", [(8, 2, 1300), (32, 8, 2049), (256, 32, 1025), (65, 13, 16384)])
def test_mixed_elections(tmp_path, hq, hkv, n):
    path = synthetic.write_cluster_table(synthetic.random_cluster_table(hq, 3, 2, 3), str(tmp_path / "table.json"))
    dev, nb, bs, d = torch.device("cuda:0"), -(-n // 128), 128, 128
    flags = _lib.SP_FLAG_LOGITS_BF16
    states = [AttentionSharing(path)._ensure_state(nb, dev) for _ in range(2)]
    n_slots = states[0].n_clusters
    gen = torch.Generator().manual_seed(hq)
    hc = torch.randint(-1, n_slots, (hq,), generator=gen, dtype=torch.int32)
    hc[::5] = torch.tensor([n_slots, -7, 2 ** 30, n_slots + 3], dtype=torch.int32).repeat(hq)[: len(hc[::5])]
    hc = hc.to(dev)
    seen = set()
    for layer in range(3):  # (no pattern is written after layer 0: layer 1 finds pivots without one)
        q, k, _ = (t[0] for t in synthetic.planted_qkv(hq, hkv, n, d, 5 + layer, device=dev, q_head_gain=1.0))
        js = _stages(AttentionSharing(path)._ensure_state(nb, dev), hc, layer, q, k, bs, flags, 4, nb, 0.9, 0.5, 1e9, 0.1)[2]["js_qa"]
        args = (q, k, bs, flags, 4, nb, 0.9, 0.5, 1e9, float(js.nanmedian()))  # half of the heads query-aware
        mask, ints, floats, _ = _stages(states[0], hc, layer, *args)
        probs = torch.zeros(hq, nb, nb, dtype=torch.float32, device=dev)
        got_mask, got_ints, got_floats = ops.select_layer(states[1], hc, layer, *args, probs, keep_floats=True)
        for want, got in zip(ints, got_ints):
            assert torch.equal(got, want)
        for name in ("js_v", "js_s"):
            assert torch.equal(got_floats[name].view(torch.int32), floats[name].view(torch.int32)), name
        assert torch.equal(got_mask, mask)
        for slab in ("info", "ratio", "pattern"):
            assert torch.equal(getattr(states[0], slab), getattr(states[1], slab)), slab
        seen |= set(ints[0].tolist())
        if layer == 1:
            maps = torch.rand(hq, nb, nb, device=dev).tril_()
            maps /= maps.sum(-1, keepdim=True)
            dense = torch.zeros_like(ints[0])
            for c in range(n_slots):  # the pivots' maps arrive only now
                h = int(states[0].info[c, 0])
                if h >= 0:
                    dense[h] = _lib.SP_DEC_DENSE
            for s in states:
                ops.pivot_update(s, hc, dense, maps, 0.9)
    assert seen >= {_lib.SP_DEC_VS, _lib.SP_DEC_DENSE, _lib.SP_DEC_SHARE, _lib.SP_DEC_QA}
