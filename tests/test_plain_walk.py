"""The plain grouped product multiplies every weight batch by the columns it belongs to, whatever the width, the format's
batch and the number of waves that share a row: the kernel's own loop (picoforge_amd/csrc/pf_plain_walk.h) walked on the
host.  Runs without a GPU."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
WIDTHS = list(range(128, 2816 + 1, 128))   # half a 256-batch (a padded Q2_K row's logical width) included


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    exe = tmp_path_factory.mktemp("walk") / "check_plain_walk"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-o", str(exe), str(ROOT / "tests" / "check_plain_walk.cpp")], check=True)
    return exe


@pytest.mark.parametrize("batch_cols", [128, 256], ids=["q8_0-mxfp4", "q2_k"])
@pytest.mark.parametrize("parts", [1, 4], ids=["whole", "split"])
def test_every_batch_meets_its_own_columns(walker, batch_cols, parts):
    for width in WIDTHS:
        run = subprocess.run([str(walker), str(width), str(batch_cols), str(parts)], capture_output=True, text=True)
        assert run.returncode == 0, f"width {width}: {run.stderr}"
        assert int(run.stdout) == -(-width // batch_cols)
