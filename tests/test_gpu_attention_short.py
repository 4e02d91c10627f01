"""GPU parity of the short-prompt attention kernel with the fp32 masked-attention oracle (bounds and their derivation:
test_gpu_attention.py; the block-average maps add the probabilities as rounded to bf16, 2^-8 relative each, and are compared
to 2^-8)."""

import numpy as np
import pytest
import torch

from oracle import shareprefill_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_REL = 2e-2, 2.5e-3


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,n", [(8, 8, 1), (8, 1, 65), (16, 4, 130), (4, 2, 640), (7, 1, 1111),
                                      (32, 8, 2048),   # whole blocks
                                      (32, 8, 2177),   # ragged by one token
                                      (3, 1, 8300)])   # more than one mask word per row
def test_short_attention_matches_oracle(gpu_device, hq, hkv, n, d):
    """Random masks with dense heads among them, whose maps the kernel writes; logits that grow along the row for the last
    head, so that the running max has to move."""
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


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,n", [(8, 8, 257),    # no groups, a last block of one token
                                      (24, 3, 700),   # heads rotate over the XCDs; groups of eight
                                      (14, 2, 1153),  # they do not; groups of seven
                                      (40, 8, 8321)])  # two mask words a row, groups of five
def test_rows_whose_first_kept_block_is_not_the_first(gpu_device, hq, hkv, n, d):
    """A row's first tile is asked for as block 0's before its mask is there: rows that keep that block and rows that do not,
    some of them keeping nothing but their own, some nothing in their first mask word; keys and values in rows wider than the head."""
    from shareprefill_amd import ops

    gen = torch.Generator().manual_seed(n + d)
    mk = lambda h, width: torch.randn(n, h, width, generator=gen).to(torch.bfloat16)[..., :d].transpose(0, 1)
    q, k, v = mk(hq, d), mk(hkv, d + 8), mk(hkv, 2 * d)
    nb = -(-n // 128)
    rng = np.random.default_rng(n)
    mask = np.tril(rng.random((hq, nb, nb)) < 0.3)
    mask[:, 1::2, 0] = False
    mask[::3, nb // 2, :] = False
    mask[1::3, -1, :min(64, nb - 1)] = False
    mask[:, np.arange(nb), np.arange(nb)] = True
    ref, _ = O.masked_attention(q, k, v, mask, 128, d ** -0.5)
    bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
    on_gpu = lambda t: t.transpose(0, 1).to(gpu_device).transpose(0, 1)
    wide = lambda t, width: torch.nn.functional.pad(on_gpu(t).transpose(0, 1), (0, width - d), value=float("nan"))[..., :d].transpose(0, 1)
    out = ops.short_attention(on_gpu(q), wide(k, d + 8), wide(v, 2 * d), bits, d ** -0.5).transpose(0, 1).float().cpu()
    ref = ref.float()
    assert (out - ref).abs().max().item() <= MAX_ABS
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= MEAN_REL


@pytest.mark.parametrize("hq,hkv,n,d", [(6, 2, 1, 64), (6, 2, 1111, 128), (6, 6, 2177, 64), (32, 8, 2048, 128),
                                        (32, 8, 2177, 128), (3, 1, 8300, 128)])
def test_pivot_patterns_in_the_attention_launch(gpu_device, hq, hkv, n, d):
    """State, maps and outputs of the launch that also updates the pivots' state equal those of two calls, to the bit,
    with several dense heads of a cluster, a dense head without one and clusters without a dense head; counters and
    accumulators serve a second call."""
    from shareprefill_amd import ops

    nb = -(-n // 128)
    rng = np.random.default_rng(n + d)
    hc = torch.tensor([(-1, 0, 1, 2, 0, 2)[h % 6] for h in range(hq)], dtype=torch.int32, device=gpu_device)
    dense = np.array([h % 6 in (0, 1, 4) or h == 2 for h in range(hq)])
    decision = torch.where(torch.from_numpy(dense), O.DEC_DENSE, O.DEC_VS).to(torch.int32).to(gpu_device)
    states = [ops.ClusterState(3, nb, gpu_device, keep_maps=True) for _ in range(2)]
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    for rep in range(2):
        mask = np.tril(rng.random((hq, nb, nb)) < 0.4)
        mask[:, np.arange(nb), np.arange(nb)] = True
        mask[dense] = np.tril(np.ones((nb, nb), dtype=bool))
        bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
        q, k, v = (torch.randn(h, n, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h in (hq, hkv, hkv))
        cols, dists = (torch.from_numpy(rng.random((3, nb)) < 0.3).to(gpu_device) for _ in range(2))
        avgs = [torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device) for _ in range(2)]
        for state in states:
            state.cols.copy_(cols)
            state.dists.copy_(dists)
        out = ops.short_attention(q, k, v, bits, d ** -0.5, decision, avgs[0])
        ops.pivot_update(states[0], hc, decision, avgs[0], 0.9)
        got = ops.short_attention(q, k, v, bits, d ** -0.5, decision, avgs[1], pivot=(states[1], hc, 0.9))
        assert torch.equal(got, out) and torch.equal(avgs[0], avgs[1])
        for slab in ("info", "pattern", "accum", "avg_map"):  # (the third cluster's map is never written)
            assert torch.equal(getattr(states[0], slab)[:2], getattr(states[1], slab)[:2]), slab
        assert torch.equal(states[0].ratio.view(torch.int64), states[1].ratio.view(torch.int64))
        assert states[1].info[:, 1].tolist() == [1, 1, 0]
        assert not states[1].accum.any() and not states[1].info[:, 5].any()


@pytest.mark.parametrize("hq,hkv,n,d", [(6, 2, 1111, 128), (72, 8, 1111, 64), (70, 2, 1025, 128)])
def test_block_sums_for_as_many_heads_as_can_be_pivots(gpu_device, hq, hkv, n, d):
    """Maps, with room for exactly the dense heads, equal those with room for all heads (also of more heads than a wave has
    lanes); a dense head there is no room for gets NaN and updates no pivot, the others are as they were."""
    from shareprefill_amd import ops

    nb = -(-n // 128)
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    q, k, v = (torch.randn(h, n, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h in (hq, hkv, hkv))
    dense = np.arange(hq) % 5 == 1
    decision = torch.where(torch.from_numpy(dense), O.DEC_DENSE, O.DEC_VS).to(torch.int32).to(gpu_device)
    mask = ops.bool_to_mask(torch.ones(nb, nb, dtype=torch.bool).tril().expand(hq, nb, nb)).to(gpu_device)
    room = int(dense.sum())
    avgs = [torch.zeros(hq, nb, nb, dtype=torch.float32, device=gpu_device) for _ in range(3)]
    hc = torch.arange(hq, dtype=torch.int32, device=gpu_device)
    state = ops.ClusterState(hq, nb, gpu_device, keep_maps=False)
    outs = [ops.short_attention(q, k, v, mask, d ** -0.5, decision, avgs[0]),
            ops.short_attention(q, k, v, mask, d ** -0.5, decision, avgs[1], max_pivots=room),
            ops.short_attention(q, k, v, mask, d ** -0.5, decision, avgs[2], max_pivots=room - 1, pivot=(state, hc, 0.9))]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert torch.equal(avgs[0], avgs[1]) and not avgs[0].isnan().any()
    last = int(np.nonzero(dense)[0][-1])
    assert avgs[2][last].isnan().any()
    others = torch.arange(hq, device=gpu_device) != last
    assert torch.equal(avgs[0][others], avgs[2][others])
    want = torch.from_numpy(dense).to(gpu_device) & others
    assert torch.equal(state.info[:, 1] != 0, want)
    ops.short_attention(q, k, v, mask, d ** -0.5, torch.zeros_like(decision), avgs[1], max_pivots=0)


def test_a_layer_keeps_block_sums_of_its_possible_pivots_only(gpu_device, tmp_path):
    """32 heads of 64 channels at 32768 tokens: what stays allocated for their maps is that of the long-prompt kernel for
    as many heads as the layer has shared clusters, and nothing in a layer without one."""
    import json
    import types

    from shareprefill_amd import AttentionSharing, _lib, ops, shareprefill_attention_forward, synthetic

    hq, hkv, n, d = 32, 8, 32768, 64
    path = tmp_path / "table.json"  # layer 0: two shared clusters; layer 1: none
    path.write_text(json.dumps({"clusters": {"a": [[0, h] for h in range(9)], "b": [[0, h] for h in range(9, 14)],
                                             "c": [[1, h] for h in range(32)]}, "shared_clusters": ["a", "b"]}))
    cfg = types.SimpleNamespace(block_size=128, min_budget=1024, max_budget=None, pattern_threshold=0.9, similarity_threshold=0.5,
                                fallback_threshold=0.9, queryaware_threshold=0.0)
    sharing = AttentionSharing(str(path))
    qkv = synthetic.planted_qkv(hq, hkv, n, d, 1, device=gpu_device, q_head_gain=1.0)
    held = lambda: sum(buf.numel() for key, buf in ops._workspaces.items() if key[0] == "attn_short")
    torch.cuda.synchronize()
    ops.release_workspaces()
    for layer, pivots in ((1, 0), (0, 2)):
        mod = types.SimpleNamespace(config=cfg, attention_sharing=sharing, layer_idx=layer, scaling=d ** -0.5)
        shareprefill_attention_forward(mod, *qkv, None, scaling=d ** -0.5)
        assert int((sharing.plans[-1].decision == _lib.SP_DEC_DENSE).sum()) == pivots
        assert held() <= pivots * _lib.load().sp_attn_pivot_scratch_bytes(n, 128)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,n", [(8, 2, 130), (6, 2, 700), (32, 8, 2048), (3, 1, 6177)])
def test_short_and_long_prompt_kernels_give_the_same_bits(gpu_device, hq, hkv, n, d):
    """Both walk a row's blocks in steps of 32 keys and move the running max by the same rule, so which of them a prompt's
    length chooses does not show in its output; logits that grow along the row make the max move often."""
    from shareprefill_amd import ops

    nb = -(-n // 128)
    gen = torch.Generator(device=gpu_device).manual_seed(n + d)
    q, k, v = (torch.randn(h, n, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h in (hq, hkv, hkv))
    k[-1] *= (1 + 9 * torch.arange(n, device=gpu_device) / n)[:, None].to(torch.bfloat16)
    mask = np.tril(np.random.default_rng(n).random((hq, nb, nb)) < 0.4)
    mask[:, np.arange(nb), np.arange(nb)] = True
    bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
    short = ops.short_attention(q, k, v, bits, d ** -0.5)
    wide = (torch.nn.functional.pad(t, (0, 128 - d)) for t in (q, k, v))
    long = ops.block_sparse_attention(*wide, bits, 128, d ** -0.5, half_channels=d == 64)[..., :d]
    assert torch.equal(short, long)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("past", [0, 1])
def test_dense_prompts_on_both_sides_of_the_line(gpu_device, tmp_path, d, past):
    """A prompt within the minimum budget, at the last length the short-prompt kernel takes it and at the first it does
    not: output on the dense mask, cleared maps."""
    import types

    from shareprefill_amd import AttentionSharing, _lib, ops, shareprefill_attention_forward, synthetic

    n = _lib.load().sp_short_attn_max_dense_tokens(d) + past
    path = synthetic.write_cluster_table(synthetic.random_cluster_table(2, 1, 1, 3), str(tmp_path / "table.json"))
    cfg = types.SimpleNamespace(block_size=128, min_budget=65536, max_budget=None, pattern_threshold=0.9, similarity_threshold=0.5,
                                fallback_threshold=0.9, queryaware_threshold=0.1)
    qkv = synthetic.planted_qkv(2, 1, n, d, 1, device=gpu_device, q_head_gain=1.0)
    mod = types.SimpleNamespace(config=cfg, attention_sharing=AttentionSharing(path), layer_idx=0, scaling=d ** -0.5)
    out, maps = shareprefill_attention_forward(mod, *qkv, None, scaling=d ** -0.5)
    nb = -(-n // 128)
    mask = ops.bool_to_mask(torch.ones(nb, nb, dtype=torch.bool).tril().expand(2, nb, nb)).to(gpu_device)
    want = ops.block_sparse_attention(*(torch.nn.functional.pad(t[0], (0, 128 - d)) for t in qkv), mask, 128, d ** -0.5,
                                      half_channels=d == 64)[..., :d]
    assert torch.equal(out[0], want) and not maps.any() and maps.shape == (1, 2, nb, nb)


@pytest.mark.parametrize("hq,hkv,n", [(3, 1, 65537),  # more than eight mask words a row
                                      (2, 1, 131072)])
def test_long_prompts_of_64_channels_have_the_long_prompt_kernels_bits(gpu_device, hq, hkv, n):
    from shareprefill_amd import ops

    d, nb = 64, -(-n // 128)
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    q, k, v = (torch.randn(h, n, d, generator=gen, device=gpu_device).to(torch.bfloat16) for h in (hq, hkv, hkv))
    mask = np.tril(np.random.default_rng(n).random((hq, nb, nb)) < 4.0 / nb)
    mask[:, np.arange(nb), np.arange(nb)] = True
    bits = ops.bool_to_mask(torch.from_numpy(mask)).to(gpu_device)
    wide = (torch.nn.functional.pad(t, (0, 128 - d)) for t in (q, k, v))
    long = ops.block_sparse_attention(*wide, bits, 128, d ** -0.5, half_channels=True)[..., :d]
    assert torch.equal(ops.short_attention(q, k, v, bits, d ** -0.5), long)


@pytest.mark.parametrize("hq,hkv,n,d,pattern", [(8, 2, 6657, 128, 0.9), (8, 2, 10241, 128, 0.65), (4, 2, 32769, 64, 0.95),
                                                (4, 2, 65537, 64, 0.99)])
def test_steady_layers_take_the_short_prompt_kernel_further(gpu_device, tmp_path, monkeypatch, hq, hkv, n, d, pattern):
    """Three layers, the first of which opens every cluster: the others are the short-prompt kernel's up to a line that depends on the
    coverage; outputs, maps and state are those of the persistent kernel in every layer."""
    import types

    from shareprefill_amd import AttentionSharing, _lib, ops, shareprefill_attention_forward, shareprefill_attn, synthetic

    lib = _lib.load()
    further = lib.sp_short_attn_max_tokens(d) < n <= lib.sp_short_attn_max_steady_tokens(d, pattern)
    assert further == (n != 65537)
    path = synthetic.write_cluster_table(synthetic.random_cluster_table(hq, 2, 3, n), str(tmp_path / "table.json"))
    cfg = types.SimpleNamespace(block_size=128, min_budget=1024, max_budget=None, pattern_threshold=pattern, similarity_threshold=0.5,
                                fallback_threshold=1e9, queryaware_threshold=0.1)
    qkv = [synthetic.planted_qkv(hq, hkv, n, d, 7 + layer, device=gpu_device, q_head_gain=1.0) for layer in range(3)]
    calls = []
    short = ops.short_attention
    monkeypatch.setattr(ops, "short_attention", lambda *a, **kw: calls.append(len(results)) or short(*a, **kw))
    passes = []
    for steady in (True, False):
        if not steady:
            monkeypatch.setattr(shareprefill_attn, "_short_in_steady_layers", lambda *a: False)
        sharing, results = AttentionSharing(path), []
        assert [sharing.opens_cluster(layer, hq) for layer in range(3)] == [True, False, False]
        for layer in range(3):
            mod = types.SimpleNamespace(config=cfg, attention_sharing=sharing, layer_idx=layer, scaling=d ** -0.5)
            results.append(shareprefill_attention_forward(mod, *qkv[layer], None, scaling=d ** -0.5))
        passes.append((results, sharing._state))
    assert calls == ([1, 2] if further else [])
    (got, state), (want, state_want) = passes
    for (out, maps), (out_want, maps_want) in zip(got, want):
        assert torch.equal(out, out_want) and torch.equal(maps, maps_want)
    assert torch.equal(state.info, state_want.info) and torch.equal(state.pattern, state_want.pattern)


@pytest.mark.parametrize("hq,hkv,n,d,pattern", [(8, 2, 6913, 128, 0.9), (2, 1, 65665, 64, 0.95), (2, 1, 131072, 64, 0.95)])
def test_a_steady_layer_that_elects_after_all(gpu_device, tmp_path, monkeypatch, hq, hkv, n, d, pattern):
    """A first layer whose heads are all query-aware elects no pivot, the second, which opens no cluster, does: in the short-prompt
    kernel, up to its longest rows, with the persistent one's output.  A map's entries are differences of running sums of weights that
    come to at most 1 each query, kept in fp32: 2^-20 from the persistent kernel's, which moves a block in or out of a pattern here and
    there.  Both kernels keep block sums in one place, which is no larger than the persistent kernel's alone."""
    import types

    from shareprefill_amd import AttentionSharing, _lib, ops, shareprefill_attention_forward, shareprefill_attn, synthetic

    lib = _lib.load()
    assert lib.sp_short_attn_max_tokens(d) < n <= lib.sp_short_attn_max_steady_tokens(d, pattern)
    path = synthetic.write_cluster_table(synthetic.random_cluster_table(hq, 2, 2, n), str(tmp_path / "table.json"))
    qkv = [synthetic.planted_qkv(hq, hkv, n, d, 7 + layer, device=gpu_device, q_head_gain=1.0) for layer in range(2)]
    calls = []
    short = ops.short_attention
    monkeypatch.setattr(ops, "short_attention", lambda *a, **kw: calls.append(len(results)) or short(*a, **kw))
    passes, held = [], []
    for steady in (True, False):
        if not steady:
            monkeypatch.setattr(shareprefill_attn, "_short_in_steady_layers", lambda *a: False)
        sharing, results = AttentionSharing(path), []
        torch.cuda.synchronize()
        ops.release_workspaces()
        for layer in range(2):
            cfg = types.SimpleNamespace(block_size=128, min_budget=1024, max_budget=None, pattern_threshold=pattern, similarity_threshold=0.5,
                                        fallback_threshold=1e9, queryaware_threshold=0.0 if layer else 2.0)
            mod = types.SimpleNamespace(config=cfg, attention_sharing=sharing, layer_idx=layer, scaling=d ** -0.5)
            out, maps = shareprefill_attention_forward(mod, *qkv[layer], None, scaling=d ** -0.5)
            results.append((out, maps, sharing.plans[-1].decision))
        passes.append((results, sharing._state))
        held.append(sum(buf.numel() for key, buf in ops._workspaces.items() if key[0].startswith("attn_")))
    assert calls == [1] and held[0] == held[1]
    (got, state), (want, state_want) = passes
    assert (got[0][2] == _lib.SP_DEC_QA).all() and (got[1][2] == _lib.SP_DEC_DENSE).any()
    for (out, maps, decision), (out_want, maps_want, decision_want) in zip(got, want):
        assert torch.equal(decision, decision_want) and torch.equal(out, out_want)
        assert (maps - maps_want).abs().max().item() <= 2.0 ** -20
    assert torch.equal(state.info, state_want.info) and (state.info[:, 1] != 0).any()
    nb = -(-n // 128)
    moved = ops.mask_to_bool(state.pattern, nb) != ops.mask_to_bool(state_want.pattern, nb)
    assert moved.float().mean().item() <= 1e-4


@pytest.mark.parametrize("n", [65665, 131072])  # 514 and 1024 blocks
def test_pivot_patterns_of_the_longest_rows(gpu_device, n):
    test_pivot_patterns_in_the_attention_launch(gpu_device, 3, 1, n, 64)
