"""The tile map of the dense workgroup tiles and the hyper-connection mix-up
(csrc/q38m_tiles.h), walked on the host (tests/tile_map_check.cpp): each tile
once, and only grids that a launch can take."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qwen3.8-flash-next-dual-gpu_amd", "csrc")


def test_tile_map(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "tile_map_check.cpp")], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout
    assert int(re.search(r"maps (\d+)", run.stdout).group(1)) > 1000
