"""The index rules of csrc/tile_index.h, checked on the host for every width up to 640."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rows_read_by_a_k_major_tile_stay_inside_the_operand(tmp_path):
    exe = str(tmp_path / "tile_index_test")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", os.path.join(HERE, "tile_index_test.cpp"), "-o", exe], check=True)
    done = subprocess.run([exe], capture_output=True, text=True)
    assert done.returncode == 0 and done.stdout.startswith("ok"), done.stdout
