"""Gangs of the persistent attention kernel at the edges of their sizes and of the ranked range: every (row, head) exactly once,
by the check and the bounds of test_gpu_attention_schedule.py."""

import pytest
from test_gpu_attention_schedule import test_every_row_once_and_pivots_in_their_slots as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,n,max_pivots", [
    (6, 1, 10007, 2),     # three gangs of 14 of 40 pairs: two padding tickets per head
    (2, 1, 16384, 0),     # 64 pairs: the last length with gangs of at most 16
    (3, 3, 16385, 1),     # 65 pairs in three gangs of 22
    (2, 2, 32768, 1),     # the last ranked length
    (256, 8, 8321, 3),    # every head the kernel takes: 768 gangs
])
def test_gangs(gpu_device, hq, hkv, n, max_pivots):
    check(gpu_device, hq, hkv, n, max_pivots)
