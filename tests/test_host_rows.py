"""The host side of longer host-pointer forwards on the CPU, under the sanitizers.

tests/check_host_rows.cpp drives picoforge_amd/csrc/pf_host_rows.h (the ring of page-locked pieces, the copy crew, slots and
their hand-over) with a thread in the place of the GPU's stream and several callers at once: once with AddressSanitizer and
UndefinedBehaviorSanitizer and once with ThreadSanitizer."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.parametrize("sanitizer", ["address,undefined", "thread"])
def test_rows_through_the_ring_by_several_callers(tmp_path, sanitizer):
    exe = tmp_path / "check_host_rows"
    subprocess.run(["g++", "-std=c++17", "-g", "-O1", f"-fsanitize={sanitizer}", "-fno-sanitize-recover=all", "-pthread", "-o", str(exe),
                    str(ROOT / "tests" / "check_host_rows.cpp")], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=240)
    print(run.stdout, run.stderr)
    assert run.returncode == 0, run.stderr
    assert run.stdout.startswith("0 faults")


def test_page_locked_memory_of_a_ring(tmp_path):
    """A workspace of more than 64 tokens holds 4 MB of it."""
    source = f'#include "{ROOT}/picoforge_amd/csrc/pf_host_rows.h"\nstatic_assert(PF_RING_SLOTS * PF_RING_BYTES == (size_t)4 << 20, "the ring");\n'
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-x", "c++", "-"], input=source, text=True, check=True)
