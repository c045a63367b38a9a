"""Requests whose words, admitted and finished together, are too many for one launch of a
workgroup per 256 of them (fills) or 512 (hashes)."""
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def test_more_words_than_a_launch(gpu):
    dims, n = (16, 4096, 60000), 18  # 2.5e8 words each, 2^32 with 18 of them
    thr = gpu.threshold(1, 5)
    announce(f"{n} requests of {dims}: fills and hashes in several launches")
    with gpu.World(dims, flags=gpu.DENSE) as w:
        w.fill_rain(5, thr)
        want = w.tick()
    with gpu.Server(budget_bytes=80 << 30, round_ticks=2, max_active=64) as s:
        ids = [s.submit(dims, 5, thr, 1) for _ in range(n)]
        s.drain()
        assert [s.result(i)[:2] for i in ids] == [(2, want)] * n
