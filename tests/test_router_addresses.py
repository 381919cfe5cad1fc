"""Every load that a chunk's router makes of the experts' parts lies inside their allocation, also where a workgroup takes two tiles of
32 experts and the layer has an odd number of them.

The kernel takes its addresses from picoforge_amd/csrc/pf_router_addr.h; tests/check_router_addresses.cpp compiles the same
header for the host and walks the loads of every workgroup.  Runs without a GPU."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    exe = tmp_path_factory.mktemp("router") / "check_router_addresses"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-o", str(exe), str(ROOT / "tests" / "check_router_addresses.cpp")], check=True)
    return exe


@pytest.mark.parametrize("experts", [2, 32, 33, 64, 65, 70, 96, 160, 224, 480, 500, 512, 1000])
@pytest.mark.parametrize("hidden", [256, 2560])
def test_every_load_stays_inside_the_parts(walker, experts, hidden):
    run = subprocess.run([str(walker), str(experts), str(hidden)], capture_output=True, text=True)
    print(run.stdout, run.stderr)
    assert run.returncode == 0, run.stderr
    assert int(run.stdout.split()[0]) >= 2 * ((experts + 31) // 32) * (hidden // 16) * 192
