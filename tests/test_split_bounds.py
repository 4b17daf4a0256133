"""The grid and the partial rows that the host sizes for the split the kernels
choose, over random batches (tests/native/split_bounds.cpp against
cast_amd/csrc/split_choice.hpp): a workgroup too few would leave rows unwritten
without a flag."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no C++ compiler")
def test_grid_and_partial_rows_hold_the_choice(tmp_path):
    exe = tmp_path / "split_bounds"
    cmd = ["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", f"-I{ROOT / 'cast_amd' / 'csrc'}",
           str(ROOT / "tests" / "native" / "split_bounds.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe), "60000"], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr
    word = run.stdout.split()
    assert word[-1] == "ok" and all(int(n) > 100 for n in word[1:7])   # every candidate, none fitting, left whole
    assert int(word[8]) > 0                                            # the grid is no larger than need be
