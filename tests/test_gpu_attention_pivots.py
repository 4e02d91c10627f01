"""The persistent kernel's launch that also turns the pivots' maps into patterns (sp_block_sparse_attn_pivot_fwd_bf16): outputs,
maps and state equal those of the attention call and sp_pivot_update, to the bit."""

import numpy as np
import pytest
import torch

from oracle import shareprefill_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,n,half", [
    (6, 2, 100, False),     # one block
    (12, 2, 1111, False),   # an odd number of blocks, several dense heads of a cluster
    (6, 6, 1024, True),     # channels 64.. zero
    (7, 1, 8321, False),    # ranked gangs, a ragged last block
    (2, 1, 33000, False),   # more blocks than are ranked, rows of up to 258 entries
])
def test_pivot_update_in_the_launch(gpu_device, hq, hkv, n, half):
    from shareprefill_amd import ops

    nb, d = -(-n // 128), 128
    rng = np.random.default_rng(n)
    hc = torch.tensor([(-1, 0, 1, 2, 0, 2)[h % 6] for h in range(hq)], dtype=torch.int32, device=gpu_device)
    dense = np.array([h % 6 in (0, 1, 4) or h == 2 for h in range(hq)])
    decision = torch.where(torch.from_numpy(dense), O.DEC_DENSE, O.DEC_VS).to(torch.int32).to(gpu_device)
    states = [ops.ClusterState(3, nb, gpu_device, keep_maps=True) for _ in range(2)]
    for state in states:
        state.avg_map.zero_()
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    for rep in range(2):  # (counters and accumulators serve a second call)
        mask = np.tril(rng.random((hq, nb, nb)) < 0.4)
        mask[:, np.arange(nb), np.arange(nb)] = True
        mask[dense] = np.tril(np.ones((nb, nb), dtype=bool))
        mask[dense, 1:, 0] = rep == 0  # (the second time a dense row does not start at column 0)
        bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
        q, k, v = (torch.randn(h, n, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h in (hq, hkv, hkv))
        if half:
            q, k, v = (torch.nn.functional.pad(t[..., :64], (0, 64)) for t in (q, k, v))
        cols, dists = (torch.from_numpy(rng.random((3, nb)) < 0.3).to(gpu_device) for _ in range(2))
        avgs = [torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device) for _ in range(2)]
        for state in states:
            state.cols.copy_(cols)
            state.dists.copy_(dists)
        kw = dict(decision=decision, max_pivots=hq, half_channels=half)
        out = ops.block_sparse_attention(q, k, v, bits, 128, d ** -0.5, avg_attn=avgs[0], **kw)
        ops.pivot_update(states[0], hc, decision, avgs[0], 0.9)
        got = ops.block_sparse_attention(q, k, v, bits, 128, d ** -0.5, avg_attn=avgs[1], pivot=(states[1], hc, 0.9), **kw)
        used = slice(0, 64) if half else slice(None)
        assert torch.equal(got[..., used], out[..., used]) and torch.equal(avgs[0], avgs[1])
        for slab in ("info", "pattern", "accum", "avg_map"):
            assert torch.equal(getattr(states[0], slab), getattr(states[1], slab)), slab
        assert torch.equal(states[0].ratio.view(torch.int64), states[1].ratio.view(torch.int64))
        assert not states[1].accum.any() and not states[1].info[:, 5].any()


def test_dense_heads_without_room(gpu_device):
    """A dense head beyond the room for block sums gets NaN for a map and updates no pivot, the others are as they were; through
    the entry point that does not update the pivots it takes the recomputing pass."""
    from shareprefill_amd import ops

    hq, hkv, n, d = 6, 2, 1111, 128
    nb = -(-n // 128)
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    q, k, v = (torch.randn(h, n, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h in (hq, hkv, hkv))
    dense = torch.tensor([0, 1, 1, 0, 0, 1], dtype=torch.bool)
    decision = torch.where(dense, O.DEC_DENSE, O.DEC_VS).to(torch.int32).to(gpu_device)
    mask = ops.bool_to_mask(torch.ones(nb, nb, dtype=torch.bool).tril().expand(hq, nb, nb)).to(gpu_device)
    hc = torch.arange(hq, dtype=torch.int32, device=gpu_device)
    for room in (3, 2, 0):
        state = ops.ClusterState(hq, nb, gpu_device)
        avgs = [torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device) for _ in range(2)]
        outs = [ops.block_sparse_attention(q, k, v, mask, 128, d ** -0.5, decision=decision, avg_attn=avgs[0], max_pivots=room),
                ops.block_sparse_attention(q, k, v, mask, 128, d ** -0.5, decision=decision, avg_attn=avgs[1], max_pivots=room,
                                           pivot=(state, hc, 0.9))]
        assert torch.equal(outs[0], outs[1]) and not avgs[0].isnan().any()
        served = torch.tensor([h for h in (1, 2, 5)][:room], dtype=torch.int64)
        for h in range(hq):
            if dense[h] and h not in served:
                assert avgs[1][h].isnan().sum().item() == nb * (nb + 1) // 2
            else:
                assert torch.equal(avgs[0][h], avgs[1][h])
        assert (state.info[:, 1] != 0).cpu().nonzero().reshape(-1).tolist() == served.tolist()


@pytest.mark.parametrize("n", [6657])  # (the shortest prompt of the persistent kernel)
def test_a_pivot_per_head_of_the_most_heads(gpu_device, tmp_path, n):
    """256 heads, each the only one of its cluster in the layer: more pivots than a launch keeps block sums of.  Every map is a
    mean of softmax rows (its rows sum to 1) and every cluster gets its pattern; that of a head behind the last slot covers the
    threshold like those before it."""
    import types

    from shareprefill_amd import AttentionSharing, _lib, ops, shareprefill_attention_forward, synthetic

    hq, hkv, d = 256, 8, 128
    assert _lib.load().sp_short_attn_max_tokens(d) == n - 1
    nb = -(-n // 128)
    table = {"clusters": {str(h): [[0, h], [1, h]] for h in range(hq)}, "shared_clusters": [str(h) for h in range(hq)]}
    sharing = AttentionSharing(synthetic.write_cluster_table(table, str(tmp_path / "table.json")))
    assert sharing.max_pivots(0, hq) == hq
    config = types.SimpleNamespace(block_size=128, min_budget=1024, max_budget=None, pattern_threshold=0.9, similarity_threshold=0.5,
                                   fallback_threshold=0.9, queryaware_threshold=0.0)  # (no head is query-aware)
    module = types.SimpleNamespace(config=config, attention_sharing=sharing, layer_idx=0, scaling=d ** -0.5)
    qkv = synthetic.planted_qkv(hq, hkv, n, d, 11, device=gpu_device, q_head_gain=1.0)
    _, maps = shareprefill_attention_forward(module, *qkv, None, scaling=module.scaling)
    assert (sharing.plans[-1].decision == _lib.SP_DEC_DENSE).all()
    # a row's masses and their total come from the same probabilities: what is left is the fp32 rounding of at most 53 sums and of
    # log2(sum) + max, of magnitude below 128 (2^-17 each)
    assert ((maps[0].double().sum(-1) - 1).abs() <= 1e-4).all()
    state = sharing._state
    assert (state.info[:, 1] != 0).all() and state.ratio.isfinite().all()
    assert torch.equal(state.avg_map, maps[0])
    kept = ops.mask_to_bool(state.pattern, nb).to(gpu_device)
    assert ((maps[0] * kept).double().sum(-1) >= 0.9 - 1e-4).all()
