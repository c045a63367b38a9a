"""Ticks of a large world's active items only, against the byte kernels: odd row and
layer counts, a row whose last word is padded and one of 64 full words, single ticks
of both parities, hashes inside a run, host edits and passes over everything between
runs."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

# over 2^29 voxels; items are 64 x 2 x 16 cells
SHAPES = [(1024, 1031, 517), (1000, 1040, 525), (4096, 257, 515), (130, 2100, 2000)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_items_match_byte_kernels(gpu, shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx)
    announce(f"item ticks {shape}")
    pool = (40, 2, 9, nz // 8, nz * 7 // 8, nx // 8, nx // 3, ny // 8, ny // 3, 3, 30)
    with gpu.World(shape) as a, gpu.World(shape, flags=gpu.DENSE) as b:
        b.fuse = False  # single byte ticks of every row quad
        for fill in (lambda w: w.fill_boxes(3, side_min=5, side_max=60), lambda w: w.fill_pillars(4, pool)):
            fill(a)
            fill(b)
            a.tick_count = b.tick_count = 2
            for k, (n, every) in enumerate(((3, 0), (4, 2), (1, 0), (5, 5), (1, 1), (12, 0), (1, 0), (30, 7), (4, 0))):
                assert list(a.run(n, every)) == list(b.run(n, every)), (k, a.tick_count)
                assert a.hash() == b.hash(), (k, a.tick_count)
                for _ in range(40):
                    x = int(rng.choice([0, 1, 63, 64, 65, nx - 1, int(rng.integers(0, nx))]))
                    y, z, v = int(rng.integers(0, ny)), int(rng.integers(0, nz)), int(rng.choice([0, 1, 2, 3, 77]))
                    a.set_voxel(x, y, z, v)
                    b.set_voxel(x, y, z, v)
                a.skip = gpu.SKIP_OFF if k == 5 else gpu.SKIP_AUTO
            assert np.array_equal(a.download(), b.download())


def test_items_mark_the_renderers_bricks(gpu):
    from fallingsand3d_amd import render as R
    from test_render_incremental_gpu import expected_maps
    shape = (1000, 1031, 525)
    announce(f"frames between item ticks {shape}")
    cam = R.orbit_camera(shape, 0.4, 1.6, 0.4, 1.5)
    with gpu.World(shape) as w:
        w.fill_pillars(4, (40, 2, 9, 65, 459, 125, 333, 130, 340, 3, 30))
        for n in (4, 1, 3, 12):  # the first frame reads every brick, the later ones what moved
            w.run(n, 0)
            R.render(w, cam, 60, 40)
            maps, want = R.render_maps(w), expected_maps(w.download())
            assert all((a == b).all() for a, b in zip(maps, want)), n
