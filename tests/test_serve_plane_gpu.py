"""The server's plane grids at row-word edges, beside byte grids (rows under 16
cells), against the oracle."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("round_ticks", [1, 8])
def test_rows_at_word_edges(gpu, O, round_ticks):
    dims = [(15, 9, 20), (16, 9, 20), (17, 3, 2), (63, 5, 31), (64, 6, 30), (65, 7, 12), (127, 4, 9), (128, 3, 40),
            (320, 2, 25), (511, 3, 5), (512, 5, 16), (16, 1, 1), (3, 2, 2)]
    seeds = np.arange(11, 11 + len(dims), dtype=np.uint64)
    thr = np.full(len(dims), O.threshold(2, 5), np.uint64)
    ticks = [5, 40, 1, 17, 33, 8, 9, 64, 16, 3, 24, 2, 7]
    announce(f"serve planes round_ticks={round_ticks}")
    with gpu.Server(budget_bytes=1 << 30, round_ticks=round_ticks, max_active=64) as s:
        for _ in range(2):  # the second stream's grids land in memory of the first's
            ids = [s.submit(d, seeds[i], thr[i], ticks[i]) for i, d in enumerate(dims)]
            s.drain()
            for i, d in enumerate(dims):
                st, h, _ = s.result(ids[i])
                want, _ = O.run(O.scene_rain(d, int(seeds[i]), int(thr[i])), 0, ticks[i], use_lut=True)
                assert st == 2 and h == O.state_hash(want), d
