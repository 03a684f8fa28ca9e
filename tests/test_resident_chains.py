"""Host check of the Kaczmarz chains kept in LDS (tests/cpp/resident_chains.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_resident_chains_only_where_columns_fit(tmp_path):
    """Tables stay as they are, and no copy of them is made, where no chain's
    columns fit; kept chains name the same columns as before."""
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    csrc = os.path.join(ROOT, "race_amd", "csrc")
    exe = str(tmp_path / "resident_chains")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-I", csrc, "-I", os.path.join(ROOT, "include"),
                           "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "cpp", "resident_chains.cpp"),
                           os.path.join(csrc, "bundle.cpp"), os.path.join(csrc, "engine.cpp"), "-o", exe],
                          timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.endswith("ok\n"), out.stdout[-2000:] + out.stderr[-2000:]
