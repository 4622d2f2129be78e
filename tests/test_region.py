"""The host's tests for buffers of one call that share memory (birdnet-neon-engine_amd/csrc/bnh_region.h, used by entry
points whose blocks may run in any order) against the bytes themselves (tests/native/region_check.cpp): window strides
of both signs, lengths and offsets in every combination of small sizes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_shared_memory_found(tmp_path):
    exe = str(tmp_path / "region_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "birdnet-neon-engine_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "region_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and "mismatches 0" in r.stdout, r.stdout + r.stderr
