"""CPU: the raster's quotients that share a divisor equal division bit for bit,
its near box holds every pixel the reference's test covers, and the rejection
by approximate barycentrics drops none (thin, huge and non-finite triangles
included)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_against_plain_division_and_a_full_scan(tmp_path):
    exe = str(tmp_path / "test_raster_geometry")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "test_raster_geometry.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
