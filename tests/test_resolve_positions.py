"""CPU check of the position arithmetic of unresolved output bytes.

The functions the emission and resolve kernels use (resolve_common.h) are
compiled for the host by tests/bounds/resolve_positions.cpp.
"""

import os
import subprocess

import pytest

from conftest import ROOT

SOURCE = os.path.join(ROOT, "tests", "bounds", "resolve_positions.cpp")
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("resolve") / "resolve_positions")
    cmd = [HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I",
           os.path.join(ROOT, "cuda-zlib_amd", "csrc"), SOURCE, "-o", out]
    proc = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-3000:]
    return out


def test_runs_are_rooted_within_a_back_reference(program):
    """However long the runs and however far back the root handed down: every
    root is 1 to 32768 bytes back, and chains have a link per 16 KiB at most."""
    proc = subprocess.run([program, "runs"], capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stdout
    assert "runs checked=125" in proc.stdout


def test_positions_past_32_bits(program):
    """Outputs around 2^32 bytes (4 GiB - 1 behind a dictionary's 32 KiB): stripes,
    roots and the last bytes' stores."""
    proc = subprocess.run([program, "stripes"], capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stdout
    assert int(proc.stdout.split("checked=")[1]) > 20000
