"""The persistent batch kernel at the edges of its three homes for a world's
planes (a wave's LDS share, a workgroup's, device memory), against the oracle."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [256, 512, 1024])
def test_worlds_at_the_lds_limits(gpu, O, threads):
    wg = 158 * 1024 * threads // 1024 // 16 - 1  # plane words of a workgroup; a wave takes fewer than `wave`
    wave = (wg + 1) // (threads // 64)
    rng = np.random.default_rng(threads)
    dims = [(64, 1, wave - 1), (64, 1, wave), (50, wave // 8, 8), (64, 1, wg), (64, 1, wg + 1), (128, 40, wg // 80 + 1),
            (1, 3, 2), (200, 5, 9), (192, 3, 4), (1000, 2, 3), (65, 33, 20)]
    announce(f"batch planes threads={threads} {dims}")
    grids = []
    for nx, ny, nz in dims:
        g = rng.choice(np.array([0, 0, 0, 1, 2, 2, 3, 3], np.uint8), size=(nz, ny, nx))
        if nx != 64:
            g[rng.random(g.shape) < 0.02] = 77
        grids.append(g)
    with gpu.Batch(dims) as b:
        b.set_config(16, threads, 1)
        b.tick_count = 3
        for i, g in enumerate(grids):
            b.upload(i, g)
        h = b.run(9)
        for i, g in enumerate(grids):
            want, _ = O.run(g, 3, 9, use_lut=True)
            assert (b.download(i) == want).all(), dims[i]
            assert int(h[i]) == O.state_hash(want), dims[i]
