"""The grouped products' launches leave no part of the chip idle while work could be cut further, and no work out:
picoforge_amd/csrc/pf_item_order.h walked on the host.  Runs without a GPU."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_how_launches_are_cut(tmp_path):
    exe = tmp_path / "check_item_order"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-o", str(exe), str(ROOT / "tests" / "check_item_order.cpp")], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
