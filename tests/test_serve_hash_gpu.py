"""Final hashes of the server's plane grids: word counts around those of a hashing
workgroup (512), several requests that finish in one round beside some that go on, and
worlds that have long come to rest when they finish."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("round_ticks", [1, 7])
def test_final_hashes(gpu, O, round_ticks):
    dims = [(64, 1, 1), (60, 7, 73), (64, 8, 64), (50, 19, 27), (130, 11, 31), (40, 33, 32), (16, 1, 9), (128, 1, 256)]
    seeds = np.arange(3, 3 + len(dims), dtype=np.uint64)
    thr = np.full(len(dims), O.threshold(2, 5), np.uint64)
    announce(f"serve hashes round_ticks={round_ticks}")
    with gpu.Server(budget_bytes=1 << 30, round_ticks=round_ticks, max_active=64) as s:
        for ticks in ([7, 7, 7, 9, 14, 14, 300, 7], [1, 2, 3, 200, 1, 2, 3, 4]):
            ids = [s.submit(d, seeds[i], thr[i], ticks[i]) for i, d in enumerate(dims)]
            s.drain()
            for i, d in enumerate(dims):
                st, h, _ = s.result(ids[i])
                want, _ = O.run(O.scene_rain(d, int(seeds[i]), int(thr[i])), 0, ticks[i], use_lut=True)
                assert st == 2 and h == O.state_hash(want), (d, ticks[i])
