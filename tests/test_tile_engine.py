"""Host check of the small-tile engine's work items: the C++ itself, compiled
with g++ (tests/native/tile_engine_check.cpp)."""
import os
import subprocess

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_small_tile_items(tmp_path):
    exe = tmp_path / "tile_engine_check"
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(NATIVE, "tile_engine_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
