"""The device's conversion to bf16 (sp_common.h: one instruction) against the integer form that the host uses, to the bit, through
block pooling: a sum of up to three bf16 values is any fp32 value (8 + 8 + 8 bits, exact), a mean of four reaches fp32 denormals."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def integer_form(x):
    """Round to nearest even on the bits; NaN keeps its upper payload bits and becomes quiet."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    nan = (u & 0x7FFFFFFF) > 0x7F800000
    return np.where(nan, (u >> 16) | 0x40, (u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def three_parts(x):
    """fp32 values as sums of three bf16 values, as bit patterns [3, len]."""
    parts, rest = [], x.astype(np.float32)
    for _ in range(3):
        top = (rest.view(np.uint32) & 0xFFFF0000).view(np.float32)
        parts.append((top.view(np.uint32) >> 16).astype(np.uint16))
        rest = np.where(np.isfinite(x), rest - np.where(np.isfinite(top), top, 0), 0).astype(np.float32)
    assert not rest.any()
    return np.stack(parts)


def pooled(parts, pool_type, device):
    """parts [tokens <= 4, len] -> bits of the pooled block of four."""
    n, d = -(-parts.shape[1] // 8) * 8, 8
    bits = np.zeros((4, n), dtype=np.uint16)
    bits[: len(parts), : parts.shape[1]] = parts
    x = torch.from_numpy(bits.view(np.int16)).to(device).view(torch.bfloat16).view(4, n // d, d).transpose(0, 1)
    from shareprefill_amd import ops

    out = ops.pool(x, 4, pool_type)
    return out.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)[: parts.shape[1]]


def test_normals_ties_overflow_and_infinities(gpu_device):
    rng = np.random.default_rng(1)
    exponent = rng.integers(20, 255, 40000).astype(np.uint32) << 23
    low = rng.integers(0, 1 << 23, 40000).astype(np.uint32)
    low[::4] = (low[::4] & ~np.uint32(0xFFFF)) | rng.choice(np.array([0x7FFF, 0x8000, 0x8001, 0], dtype=np.uint32), len(low[::4]))
    edge = np.array([0x7F7F7FFF, 0x7F7F8000, 0x7F7F8001, 0x7F7FFFFF, 0x7F7E8000, 0x7F7EFFFF, 0x7F800000, 0x3F7FFFFF, 0x3F808000,
                     0x3F818000], dtype=np.uint32)  # (the largest finite values, to infinity and below it; carries; ties both ways)
    u = np.concatenate([exponent | low, edge])
    u = np.concatenate([u, u | np.uint32(0x80000000), np.zeros(1, dtype=np.uint32)])
    x = u.view(np.float32)
    got, want = pooled(three_parts(x), "sum", gpu_device), integer_form(x)
    wrong = np.nonzero(got != want)[0]
    assert not len(wrong), [(hex(u[i]), hex(got[i]), hex(want[i])) for i in wrong[:5]]


def test_nan(gpu_device):
    bits = np.array([[0x7F81, 0x7FC0, 0x7FFF, 0xFF81, 0xFFC1, 0x7FA5]], dtype=np.uint16)  # (signalling and quiet, both signs)
    got = pooled(bits, "sum", gpu_device)
    assert np.array_equal(got, integer_form((bits[0].astype(np.uint32) << 16).view(np.float32))), [hex(g) for g in got]


def test_denormals(gpu_device):
    """Multiples of 2^-135 below and around the smallest normal number; bf16's denormals are the multiples of 2^-133."""
    k = np.concatenate([np.arange(1, 2048), (1 << 7) * 4 + np.arange(-64, 64), 4 * (1 << 7) * 2 + np.arange(-64, 64)])
    k = np.concatenate([k, -k]).astype(np.float64)
    four = (k * 2.0 ** -133).astype(np.float32)  # the sum of the four tokens
    parts = np.zeros((3, len(k)), dtype=np.uint16)
    mag, sign = np.abs(k).astype(np.int64), np.where(k < 0, 0x8000, 0).astype(np.uint16)
    for i in range(3):  # seven bits of the multiple at a time are bf16 numbers
        top = (mag >> (7 * i) & 127) << (7 * i)
        value = (top * 2.0 ** -133).astype(np.float32)
        assert not (value.view(np.uint32) & 0xFFFF).any()
        parts[i] = (value.view(np.uint32) >> 16).astype(np.uint16) | np.where(top > 0, sign, 0).astype(np.uint16)
    mean = (four.astype(np.float64) / 4).astype(np.float32)
    got, want = pooled(parts, "avg", gpu_device), integer_form(mean)
    wrong = np.nonzero(got != want)[0]
    assert not len(wrong), [(k[i], hex(got[i]), hex(want[i])) for i in wrong[:5]]
