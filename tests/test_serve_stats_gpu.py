"""The server's tick samples and busy time hold the work that its ticks are asked for: the
hash of a finished request too."""
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def test_busy_time_holds_the_final_hash(gpu):
    dims, ticks = (512, 1024, 512), 9  # the hash of 2^28 cells takes several times a tick
    announce(f"busy time of requests of {dims}")
    with gpu.Server(budget_bytes=4 << 30, round_ticks=3, max_active=4) as s:
        busy = []
        for _ in range(4):
            before = s.stats()["busy_ms"]
            s.submit(dims, 3, gpu.threshold(1, 2), ticks)
            s.drain()
            busy.append(s.stats()["busy_ms"] - before)
        tick = s.stats()["tick_p50_ms"]
        print("busy", busy, "tick", tick)
        # nine ticks and a hash of more than two ticks' time
        assert min(busy[1:]) > (ticks + 1.5) * tick
