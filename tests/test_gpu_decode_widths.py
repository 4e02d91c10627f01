"""The decode step at the head sizes and cache lengths where its instances and its launches change, by the check and the bounds of
test_gpu_decode.py."""

import pytest
from test_gpu_decode import test_decode_batch_matches_oracle as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [8, 40, 64, 72, 120, 128])
@pytest.mark.parametrize("b,hq,hkv,n", [(1, 4, 2, 1), (2, 8, 1, 129), (1, 14, 2, 1100), (1, 40, 4, 700), (2, 17, 1, 300)])
def test_head_sizes(gpu_device, b, hq, hkv, n, d):
    check(gpu_device, b, hq, hkv, n, d)


@pytest.mark.parametrize("b,n", [(1, 128), (1, 383), (1, 384), (2, 385), (16, 257)])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (12, 12, 64), (16, 1, 128), (30, 1, 32)])
def test_caches_of_a_few_tiles(gpu_device, b, n, hq, hkv, d):
    """One workgroup walks the chunks of a cache of up to three tiles: 384 keys are the last such length."""
    check(gpu_device, b, hq, hkv, n, d)
