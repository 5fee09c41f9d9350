"""Host-only checks of the tiled kernels' plan (tests/host/tile_checks.cpp): the tile and the split of K, beside timings of them all."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_and_splits(tmp_path):
    exe = str(tmp_path / "tile_checks")
    build = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{ROOT}/include", f"-I{ROOT}/nuvec_amd/csrc", f"{ROOT}/tests/host/tile_checks.cpp", "-o", exe],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-4000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and "0 failures" in run.stdout, run.stdout[-4000:] + run.stderr[-2000:]
