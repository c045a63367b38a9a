"""Rain fills, sixteen cells at a time, against the oracle: floors and rain that begin
inside a group, one and two layers, fewer than sixteen cells, odd totals, thresholds at
both ends."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (5, 3, 1), (3, 5, 2), (16, 1, 16), (17, 1, 5), (4, 4, 9), (7, 11, 13), (31, 5, 40), (64, 64, 3), (100, 41, 37)]


@pytest.mark.parametrize("thr", [0, 1 << 63, (1 << 64) - 1])
def test_fills_match_oracle(gpu, O, thr):
    seeds = np.arange(1, len(DIMS) + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
    announce(f"rain fills thr={thr:#x}")
    with gpu.Batch(DIMS) as b:
        b.fill_rain(seeds, np.full(len(DIMS), thr, np.uint64))
        for i, d in enumerate(DIMS):
            want = O.scene_rain(d, int(seeds[i]), thr)
            assert (b.download(i) == want).all(), d
            with gpu.World(d) as w:
                w.fill_rain(int(seeds[i]), thr)
                assert (w.download() == want).all(), d
