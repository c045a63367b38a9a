"""Fused pairs of dense byte ticks, which runs of two ticks take, and longer runs where
the launch shape has been set or the grid cannot be in planes: the same shapes as whole
rows per wave and x-chunks have their edges at, both start parities, runs in a graph."""
import numpy as np
import pytest

from conftest import announce
from test_fuse_gpu import SHAPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_fused_byte_pairs_match_oracle(gpu, O, shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx * 37 + ny * 5 + nz)
    g = rng.choice(np.array([0, 0, 0, 1, 2, 2, 3, 3], np.uint8), size=(nz, ny, nx))
    g[rng.random(g.shape) < 0.02] = 230
    for t0 in (6, 11):
        announce(f"fused byte pairs {shape} t0={t0}")
        for seg in (0, 64):  # with a segment set, longer runs stay on bytes too
            with gpu.World(shape, flags=gpu.DENSE) as w:
                w.fuse = True
                if seg:
                    w.segment = seg
                assert w.fuse
                w.upload(g)
                w.tick_count = t0
                cur, t = g, t0
                for n, every in ((2, 0), (2, 0), (1, 0), (2, 2)) + (((7, 0), (11, 4)) if seg else ()):
                    if n % 2:
                        w.step(n)
                        cur, _ = O.run(cur, t, n, use_lut=True)
                    else:
                        got = [int(h) for h in w.run(n, every)]
                        cur, want = O.run(cur, t, n, every, use_lut=True)
                        assert got == [int(h) for h in want][:len(got)]
                    t += n
                    assert (w.download() == cur).all(), (t0, seg, t)


def test_fused_pair_of_a_large_world(gpu):
    shape = (1024, 1024, 260)  # fused by default above 2^28 voxels
    announce(f"pairs of {shape}")
    with gpu.World(shape, flags=gpu.DENSE) as f, gpu.World(shape, flags=gpu.DENSE) as s:
        assert f.fuse
        s.fuse = False
        for w in (f, s):
            w.fill_boxes(1)
            w.tick_count = 3
            for _ in range(4):
                w.step(2)
                w.run(2, 0)
            w.step(1)
            w.step(2)
        assert f.hash() == s.hash()
