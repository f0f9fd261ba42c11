"""The maps of fo_raster.h over all grids of up to 47 x 47 macro tiles, in a CPU build."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_tile_is_taken_once(tmp_path):
    exe = str(tmp_path / "raster_cover")
    csrc = os.path.join(HERE, "..", "flashoverlap_amd", "csrc")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", csrc, os.path.join(HERE, "raster_cover.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
