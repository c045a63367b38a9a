"""What a world keeps about its bit planes between calls, on the host: list counters
and change flags through runs of every length and changes of schedule between them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plane_schedule(tmp_path):
    import fallingsand3d_amd as F
    lut = tmp_path / "lut.bin"
    F.rule_lut().tofile(lut)
    exe = tmp_path / "plane_sched_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wno-unknown-pragmas", "-o", str(exe),
                    os.path.join(ROOT, "tests", "cpp", "plane_sched_check.cpp")], check=True)
    r = subprocess.run([str(exe), str(lut)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "plane schedule checks passed" in r.stdout, r.stdout + r.stderr
