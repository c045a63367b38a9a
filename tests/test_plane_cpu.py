"""The bit-plane core on the host: every block state and variant against the
block rule table, wall slots, shifts, packing and variant planes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plane_core_against_the_rule_table(tmp_path):
    import fallingsand3d_amd as F
    lut = tmp_path / "lut.bin"
    F.rule_lut().tofile(lut)
    exe = tmp_path / "plane_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wno-unknown-pragmas", "-o", str(exe),
                    os.path.join(ROOT, "tests", "cpp", "plane_check.cpp")], check=True)
    r = subprocess.run([str(exe), str(lut)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "plane checks passed" in r.stdout, r.stdout + r.stderr
