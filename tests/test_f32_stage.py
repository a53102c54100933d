"""The staging map of the F32 projection (CPU; no device): every 16-byte unit
of a tile is stored by exactly one thread, with the columns that belong there,
also where the units are no multiple of the workgroup (two threads storing one
unit in the same step would race)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("f32") / "stage")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "qwen3.5sharp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "f32_stage_driver.cpp"), "-o", exe], check=True)
    return exe


# The tiles of linear_f32 (rows + tokens, columns / 4), then others.
@pytest.mark.parametrize("rows,c4", [(5, 640), (8, 128), (16, 64), (8, 32), (16, 32), (1, 16), (3, 48), (7, 16), (17, 80)])
def test_each_unit_staged_once(driver, rows, c4):
    assert subprocess.run([driver, str(rows), str(c4)], capture_output=True, text=True, check=True).stdout == ""
