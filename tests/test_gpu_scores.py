"""GPU parity: last-block scores (vertical / slash vectors and their block sums) against the CPU oracle."""

import pytest
import torch

from oracle import shareprefill_oracle as O
from shareprefill_amd import synthetic

pytestmark = pytest.mark.gpu


def _inputs(hq, hkv, n, seed):
    q, k, _ = synthetic.planted_qkv(hq, hkv, n, 128, seed, q_head_gain=1.0)
    return q[0], k[0]  # [H, N, D] views of token-major storage


@pytest.mark.parametrize("hq,hkv,n", [(4, 2, 1024), (8, 2, 4096), (4, 4, 1000), (2, 1, 128), (4, 1, 2304),
                                      (6, 2, 640), (7, 1, 1111)])  # odd groups: a workgroup half without a head
@pytest.mark.parametrize("bf16_logits", [False, True])
def test_lastq_scores_match_oracle(gpu_device, hq, hkv, n, bf16_logits):
    from shareprefill_amd import _lib, ops

    q, k = _inputs(hq, hkv, n, 11 + n)
    vref, sref = O.lastq_scores(q, k, 128, logits_in_input_dtype=bf16_logits)
    flags = _lib.SP_FLAG_LOGITS_BF16 if bf16_logits else 0
    vt, st, vb, sb = ops.lastq_scores(q.to(gpu_device), k.to(gpu_device), 128, flags)
    vt, st, vb, sb = vt.cpu(), st.cpu(), vb.cpu(), sb.cpu()
    # a logit that lands on the other side of a bf16 rounding boundary (MFMA vs CPU summation order) moves one
    # probability by 2^-8 relative; with fp32 logits only exp/sum rounding remains
    rtol, atol = (3e-2, 1e-6) if bf16_logits else (2e-4, 1e-8)
    assert torch.allclose(vt, vref, rtol=rtol, atol=atol)
    assert torch.allclose(st, sref, rtol=rtol, atol=atol)
    assert torch.allclose(vt.sum(-1), torch.ones(hq), atol=1e-4)
    assert torch.allclose(st.sum(-1), torch.ones(hq), atol=1e-4)
    # block sums are the right-padded 128-token sums of the token vectors the kernel itself wrote
    assert torch.allclose(vb, O.block_sum(vt, 128), rtol=1e-5, atol=1e-9)
    assert torch.allclose(sb, O.block_sum(st, 128), rtol=1e-5, atol=1e-9)


def test_lastq_scores_seeded_random_shapes(gpu_device):
    """Ragged lengths around the tile and chunk boundaries and every group size up to 8 (odd groups leave half of a
    two-head workgroup empty), fp32 logits so that the tight tolerance holds element by element."""
    import numpy as np

    from shareprefill_amd import ops

    rng = np.random.default_rng(20240607)
    lengths = [128, 129, 255, 256, 257, 383, 640, 1000, 1111, 2049, 3000, 4097, 5000, 8191]
    for case in range(24):
        hkv = int(rng.choice([1, 2, 3]))
        g = int(rng.choice([1, 2, 3, 4, 5, 7, 8]))
        n = int(rng.choice(lengths))
        hq = hkv * g
        q, k = _inputs(hq, hkv, n, 1000 + case)
        vref, sref = O.lastq_scores(q, k, 128, logits_in_input_dtype=False)
        vt, st, vb, sb = [x.cpu() for x in ops.lastq_scores(q.to(gpu_device), k.to(gpu_device), 128, 0)]
        tag = f"case {case}: hq {hq} hkv {hkv} n {n}"
        assert torch.allclose(vt, vref, rtol=2e-4, atol=1e-8), tag
        assert torch.allclose(st, sref, rtol=2e-4, atol=1e-8), tag
        assert torch.allclose(vb, O.block_sum(vt, 128), rtol=1e-5, atol=1e-9), tag
        assert torch.allclose(sb, O.block_sum(st, 128), rtol=1e-5, atol=1e-9), tag


@pytest.mark.parametrize("hq,hkv,n", [(28, 4, 10007), (32, 8, 4609), (14, 2, 20001), (7, 1, 33000),
                                      (20, 4, 10007), (8, 8, 30001)])
def test_lastq_scores_in_chunks_of_any_number_of_tiles(gpu_device, hq, hkv, n):
    """Lengths whose statistics are cut into chunks of 3 to 5 tiles, the last of them short, up to and beyond the number of chunks
    that the probabilities kernel folds itself."""
    from shareprefill_amd import ops

    q, k = _inputs(hq, hkv, n, n)
    vref, sref = O.lastq_scores(q, k, 128, logits_in_input_dtype=False)
    vt, st, _, _ = [x.cpu() for x in ops.lastq_scores(q.to(gpu_device), k.to(gpu_device), 128, 0)]
    assert torch.allclose(vt, vref, rtol=2e-4, atol=1e-8)
    assert torch.allclose(st, sref, rtol=2e-4, atol=1e-8)


@pytest.mark.parametrize("bs", [128, 64])
@pytest.mark.parametrize("hq,hkv,n", [(32, 8, 3001), (32, 8, 4097), (14, 2, 9999), (2, 1, 128)])
def test_seams_between_workgroups_do_not_depend_on_what_stood_there(gpu_device, hq, hkv, n, bs):
    """Two workgroups add to the first tile of all but the first of them: the same bits every time, over NaN as over zeros, and block
    sums that are those of the tokens."""
    from shareprefill_amd import _lib, ops

    lib = _lib.load()
    q, k = (t.to(gpu_device) for t in _inputs(hq, hkv, n, n))
    nb = -(-n // bs)
    ws = torch.empty(lib.sp_lastq_scores_workspace_bytes(n, hq, bs), dtype=torch.uint8, device=gpu_device)
    runs = []
    for fill in (0.0, float("nan"), 7.0):
        outs = [torch.full((hq, m), fill, device=gpu_device) for m in (n, n, nb, nb)]
        rc = lib.sp_lastq_scores_bf16(q.data_ptr(), k.data_ptr(), n, hq, hkv, 128, q.stride(1), q.stride(0), k.stride(1), k.stride(0), bs,
                                      _lib.SP_FLAG_LOGITS_BF16, ws.data_ptr(), ws.numel(), *(t.data_ptr() for t in outs),
                                      torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "sp_lastq_scores_bf16")
        runs.append(outs)
    for other in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], other))
    vt, st, vb, sb = (t.cpu() for t in runs[0])
    assert torch.allclose(sb, O.block_sum(st, bs), rtol=1e-5, atol=1e-9)
    assert torch.allclose(vb, O.block_sum(vt, bs), rtol=1e-5, atol=1e-9)
    assert torch.allclose(st.sum(-1), torch.ones(hq), atol=1e-4)


@pytest.mark.parametrize("bs", [64, 32, 16])
@pytest.mark.parametrize("hq,hkv,n", [(4, 2, 1024), (6, 2, 1000), (7, 1, 389), (2, 1, 128), (4, 4, 2100), (4, 2, 100),
                                      (2, 2, 64), (3, 1, 127)])  # the last three: prompts shorter than 128 tokens
def test_lastq_scores_smaller_block_sizes(gpu_device, bs, hq, hkv, n):
    """Block sizes below 128 (attention_sharing.py:127: the last bs queries): the same kernels with the rows in front
    of the last bs masked out; token vectors against the oracle with fp32 logits, block sums of bs tokens."""
    from shareprefill_amd import ops

    q, k = _inputs(hq, hkv, n, 77 + n + bs)
    vref, sref = O.lastq_scores(q, k, bs, logits_in_input_dtype=False)
    vt, st, vb, sb = [x.cpu() for x in ops.lastq_scores(q.to(gpu_device), k.to(gpu_device), bs, 0)]
    nb = -(-n // bs)
    assert vb.shape == (hq, nb) and sb.shape == (hq, nb)
    assert torch.allclose(vt, vref, rtol=2e-4, atol=1e-8)
    assert torch.allclose(st, sref, rtol=2e-4, atol=1e-8)
    assert torch.allclose(vt.sum(-1), torch.ones(hq), atol=1e-4)
    assert torch.allclose(vb, O.block_sum(vt, bs), rtol=1e-5, atol=1e-9)
    assert torch.allclose(sb, O.block_sum(st, bs), rtol=1e-5, atol=1e-9)
    # the reference's bf16 logits as well: a logit on the other side of a bf16 rounding boundary (one ulp of a logit
    # of magnitude 8 is 0.03) moves its probability by 3 %, and a slash bin near the end holds few elements
    vref, sref = O.lastq_scores(q, k, bs, logits_in_input_dtype=True)
    vt, st, _, _ = [x.cpu() for x in ops.lastq_scores(q.to(gpu_device), k.to(gpu_device), bs)]
    assert torch.allclose(vt, vref, rtol=8e-2, atol=1e-6)
    assert torch.allclose(st, sref, rtol=8e-2, atol=1e-6)


def test_lastq_scores_head_major_layout_and_determinism(gpu_device):
    from shareprefill_amd import ops

    q, k = _inputs(4, 2, 2048, 5)
    qg, kg = q.to(gpu_device), k.to(gpu_device)
    a = ops.lastq_scores(qg, kg, 128)
    b = ops.lastq_scores(qg.contiguous(), kg.contiguous(), 128)  # [H,N,D] contiguous storage
    c = ops.lastq_scores(qg, kg, 128)
    for x, y, z in zip(a, b, c):
        assert torch.equal(x, y) and torch.equal(x, z)


def test_lastq_scores_rejects_unsupported(gpu_device):
    from shareprefill_amd import ops

    q = torch.zeros(2, 256, 64, dtype=torch.bfloat16, device=gpu_device)
    with pytest.raises(NotImplementedError):
        ops.lastq_scores(q, q, 128)
    q = torch.zeros(2, 64, 128, dtype=torch.bfloat16, device=gpu_device)
    with pytest.raises(ValueError):
        ops.lastq_scores(q, q, 128)


@pytest.mark.parametrize("hq,hkv,n", [(3, 1, 128), (4, 2, 129), (14, 2, 1000), (8, 8, 2304), (7, 1, 4095)])
def test_64_channel_scores_equal_the_zero_padded_ones_bit_for_bit(gpu_device, hq, hkv, n):
    """head_dim 64 as it is against the same heads zero-padded to 128 channels (whose products and sums it shares): the
    token vectors and block sums, and the pooled block probabilities of query-aware heads."""
    from shareprefill_amd import _lib, ops

    q, k, _ = synthetic.planted_qkv(hq, hkv, n, 64, 5 + n, q_head_gain=1.0)
    q, k = q[0].to(gpu_device), k[0].to(gpu_device)
    wide = [torch.nn.functional.pad(t, (0, 64)) for t in (q, k)]
    flags = _lib.SP_FLAG_LOGITS_BF16 | _lib.SP_FLAG_SCALE_DIM(64)
    for a, b in zip(ops.lastq_scores(q, k, 128, flags), ops.lastq_scores(*wide, 128, flags)):
        assert torch.equal(a, b)
    nb = -(-n // 128)
    decision = torch.full((hq,), _lib.SP_DEC_QA, dtype=torch.int32, device=gpu_device)
    got = []
    for qx, kx in ((q, k), wide):
        mask = torch.zeros(hq, nb, (nb + 63) // 64, dtype=torch.int64, device=gpu_device)
        probs = ops.queryaware_select(ops.pool_avg(qx, 128), ops.pool_avg(kx, 128), decision, mask, 0.9, flags)
        got.append((probs, mask))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
