"""bench.py's count of the bytes that the timed ticks move: passes over the planes, and the
runs of one or two ticks that stay on bytes."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def test_plane_bytes():
    import bench
    # 20 ticks from tick 5: ten pairs, the last one split before the hash after tick 25
    assert bench.plane_passes(5, 20) == 10
    assert bench.plane_bytes(100, 5, 20) == 100 * (0.5 * 10 + 0.25 + 1.25)
    # from tick 0, not in planes: packing does the first tick
    assert bench.plane_passes(0, 4) == 3
    assert bench.plane_bytes(100, 0, 4) == 100 * (1.25 + 0.5 * 2 + 0.25 + 1.25)
    # one tick, hashed, on bytes; then the same after 50 on planes
    assert bench.plane_passes(5, 1) == 0 and bench.plane_bytes(100, 5, 1) == 200
    assert bench.plane_bytes(100, 5, 51) == bench.plane_bytes(100, 5, 50) + 200
