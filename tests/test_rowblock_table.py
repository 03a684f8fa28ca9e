"""Host checks of the row blocks' table (tests/cpp/rowblock_table.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("rowblock") / "rowblock_table")
    subprocess.check_call([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                           "-I", os.path.join(ROOT, "race_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "cpp", "rowblock_table.cpp"), "-o", exe], timeout=300)
    return exe


def run(program, what):
    out = subprocess.run([program, what], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.endswith("ok\n"), out.stdout[-2000:] + out.stderr[-2000:]


def test_loaded_columns_lie_in_their_own_matrix(program):
    """Empty rows at the start, in the middle and at the end of a matrix of a
    batch: no thread of a block reads x past its own matrix."""
    run(program, "columns")


def test_growing_batch_moves_its_entries_seldom(program):
    """Adding matrix after matrix takes time in proportion to their entries."""
    run(program, "growth")
