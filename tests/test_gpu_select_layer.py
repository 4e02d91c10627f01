"""The one-call selection of a layer gives the bits of the stage-by-stage calls: both run the same device code, so
every float, budget, decision, mask word and state slab must be equal."""

import pytest
import torch

from shareprefill_amd import AttentionSharing, _lib, ops, synthetic

pytestmark = pytest.mark.gpu


def _stages(state, hc, layer, q, k, bs, flags, minb, maxb, pt, st, ft, qt):
    vert_tok, slash_tok, vert_blk, slash_blk = ops.lastq_scores(q, k, bs, flags)
    nv, ns = ops.cover_budgets(vert_tok, slash_tok, bs, pt, minb, maxb)
    kbar = ops.pool_avg(k, bs)
    avg_qk, js_qa, use_qa = ops.queryaware_test(q, kbar, vert_blk, bs, qt, flags)
    decision, js_v, js_s, nv_f, ns_f = ops.share_decide(state, hc, layer, vert_blk, slash_blk, use_qa, nv, ns, minb, st, ft)
    mask = ops.build_mask(state, hc, decision, vert_blk, slash_blk, nv_f, ns_f)
    qbar = ops.pool_avg(q, bs, tail_mode=_lib.SP_POOL_TAIL_RESCALE, head_enable=use_qa)
    probs = ops.queryaware_select(qbar, kbar, decision, mask, pt, flags)
    floats = dict(vert_tok=vert_tok, slash_tok=slash_tok, vert_blk=vert_blk, slash_blk=slash_blk, avg_qk=avg_qk,
                  js_qa=js_qa, js_v=js_v, js_s=js_s, kbar=kbar)
    return mask, (decision, nv, ns, nv_f, ns_f), floats, probs


# one block past the minimum, ragged tails, odd groups, 64 channels, small blocks, more than 32 score chunks (folded by a
# launch of their own), more than 256 blocks and more than 131072 tokens (budgets and selection in several launches)
@pytest.mark.parametrize("hq,hkv,d,n,bs", [
    (8, 2, 128, 1025, 128), (32, 8, 128, 3001, 128), (6, 2, 64, 2049, 128), (28, 4, 128, 4096, 128),
    (1, 1, 128, 128, 128), (5, 5, 64, 6177, 128), (4, 2, 128, 1111, 64), (4, 1, 64, 777, 16),
    (3, 1, 128, 33000, 128), (1, 1, 64, 131201, 128)])
@pytest.mark.parametrize("queryaware", [0.0, 0.1, 1e9])
def test_one_call_equals_the_stages(tmp_path, hq, hkv, d, n, bs, queryaware):
    path = synthetic.write_cluster_table(synthetic.random_cluster_table(hq, 2, 2, 3), str(tmp_path / "table.json"))
    dev, nb = torch.device("cuda:0"), -(-n // bs)
    flags = _lib.SP_FLAG_LOGITS_BF16 | _lib.SP_FLAG_SCALE_DIM(d)
    sharing = [AttentionSharing(path) for _ in range(2)]
    states = [s._ensure_state(nb, dev) for s in sharing]
    hc = sharing[0]._head_cluster_tensor(0, hq, dev)
    for layer in range(2):  # the layer that elects pivots, then one that finds them
        q, k, _ = (t[0] for t in synthetic.planted_qkv(hq, hkv, n, d, 5 + layer, device=dev, q_head_gain=1.0))
        args = (q, k, bs, flags, 4, min(nb, 10 ** 6), 0.9, 0.5, 1e9, queryaware)
        mask, ints, floats, probs = _stages(states[0], hc, layer, *args)
        got_probs = torch.zeros(hq, nb, nb, dtype=torch.float32, device=dev)
        avg = torch.full((hq, nb, nb), 7.0, dtype=torch.float32, device=dev)
        got_mask, got_ints, got_floats = ops.select_layer(states[1], hc, layer, *args, got_probs, avg_attn=avg, keep_floats=True)
        for name, want in floats.items():
            assert torch.equal(got_floats[name].view(torch.int16), want.view(torch.int16)), name
        for want, got in zip(ints, got_ints):
            assert torch.equal(got, want)
        assert torch.equal(got_mask, mask)
        assert not avg.any()
        qa = ints[0] == _lib.SP_DEC_QA
        assert torch.equal(got_probs[qa], probs[qa])
        # the inputs are such that every branch of the launches is taken: all heads query-aware (the divergence of a single
        # block may be NaN), or one pivot per shared cluster, then all of a cluster's heads sharing its pattern
        if queryaware == 1e9:
            assert qa.all() or nb == 1
        else:
            assert not qa.any() or nb == 1
            shared = hc >= 0
            if layer == 0:
                assert sorted(hc[ints[0] == _lib.SP_DEC_DENSE].tolist()) == sorted(set(hc[shared].tolist()))
            else:
                assert (ints[0][shared] == _lib.SP_DEC_SHARE).all()
        for slab in ("info", "ratio", "pattern", "accum"):
            assert torch.equal(getattr(states[0], slab), getattr(states[1], slab)), slab
        for slot in (states[0].info[:, 0] >= 0).nonzero().flatten().tolist():
            for slab in ("vert", "slash", "cols", "dists"):
                assert torch.equal(getattr(states[0], slab)[slot], getattr(states[1], slab)[slot]), slab
        # a map for every pivot, so that the next layer finds a pattern
        maps = torch.rand(hq, nb, nb, device=dev).tril_()
        maps /= maps.sum(-1, keepdim=True)
        for s in states:
            ops.pivot_update(s, hc, ints[0], maps, 0.9)
