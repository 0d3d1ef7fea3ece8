"""Calls that stage values in pinned host memory, where that memory cannot be
had (tests/integration/host_limits.cpp refuses hipHostMalloc): the same values
through ordinary memory.  Set-up and steps pin none, and the downloads of two
contexts in turn share one piece.  A permeability solve whose steps replay a
graph gives the same k where no graph can be made."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

import lbamd

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "badchimp-cpp_amd", "lib")


@pytest.fixture(scope="module")
def limits(tmp_path_factory):
    """run(mode, buffers): (stdout, values) of the program."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    lbamd.lib()  # built
    tmp = tmp_path_factory.mktemp("limits")
    exe = str(tmp / "host_limits")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "integration", "host_limits.cpp"), "-o", exe, "-L", LIB,
                    "-lbadchimp_amd", "-Wl,-rpath," + LIB, "-L/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib",
                    "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64", "-ldl"], check=True, capture_output=True, timeout=100)

    def run(mode, buffers="pageable"):
        out = str(tmp / (mode + buffers))
        r = subprocess.run([exe, mode, out, buffers], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-2000:])
        return r.stdout, np.fromfile(out)
    return run


def test_values_without_pinned_memory(gpu_available, limits):
    """Fields of one and two phases, and packed and unpacked halos and colours."""
    text, pinned = limits("pin")
    assert "pinned before a download 0\n" in text and "pinned for fields 1\n" in text, text
    text, plain = limits("nopin")
    assert int(re.search(r"pinned (\d+),", text).group(1)) >= 5, text
    assert pinned.size > 20000 and np.abs(pinned).max() > 0.1 and np.isfinite(pinned).all()
    assert np.array_equal(pinned, plain)


@pytest.mark.parametrize("buffers", ["pinned", "device", "managed"])
def test_halo_buffers_in_any_memory(gpu_available, limits, buffers):
    """Packs and unpacks in the caller's pinned, device and managed memory."""
    assert np.array_equal(limits("pin", buffers)[1], limits("pin")[1])


def test_solve_without_graphs(gpu_available, limits):
    text, graphed = limits("pin")
    assert int(re.search(r"graphs (\d+)", text).group(1)) == 2, text  # one per starting buffer
    text, plain = limits("nograph")
    assert int(re.search(r"graphs (\d+)", text).group(1)) == 1, text
    assert np.array_equal(graphed, plain)
