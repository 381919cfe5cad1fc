"""A ring piece's number reaches the host after the rows of every workgroup that wrote them, by the memory model.

tests/check_piece_order.cpp runs the steps of picoforge_amd/csrc/pf_piece_order.h, which pf_k_copy_piece is made of, on vector clocks.
Runs without a GPU."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = tmp_path_factory.mktemp("piece") / "check_piece_order"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", str(exe), str(ROOT / "tests" / "check_piece_order.cpp")], check=True)
    return exe


@pytest.mark.parametrize("out", [0, 1])
@pytest.mark.parametrize("workgroups", [1, 2, 31, 32])
def test_the_number_comes_after_every_workgroups_rows(model, workgroups, out):
    run = subprocess.run([str(model), str(workgroups), str(out)], capture_output=True, text=True, timeout=60)
    print(run.stdout, run.stderr)
    assert run.returncode == 0 and run.stdout.startswith("0 unordered")
