"""The planners against their kernels' limits, without a GPU: a driver
(tests/c_api/host_passes.cpp) plans passes through the library's internal
headers and checks what their launches would ask for."""
import os
import shutil
import subprocess

import pytest

from decomp_mpi_amd import build as B


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    if not os.path.exists(B.LIB):
        B.build()
    exe = str(tmp_path_factory.mktemp("passes") / "host_passes")
    r = subprocess.run(["g++", *B.HOST_FLAGS, "-o", exe, os.path.join(B.ROOT, "tests", "c_api", "host_passes.cpp"), B.LIB,
                        f"-Wl,-rpath,{os.path.dirname(B.LIB)}", f"-L{B.ROCM}/lib", f"-Wl,-rpath,{B.ROCM}/lib",
                        "-lamdhip64"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def run(driver, check):
    r = subprocess.run([driver, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("OK\n"), r.stdout[-4000:] + r.stderr[-2000:]


def test_workgroup_lds(driver):
    """No pass asks for more than the 160 KiB of LDS that a workgroup has."""
    run(driver, "lds")


def test_table_bytes(driver):
    """A pass's tables stay bounded with more rank positions than LDS holds."""
    run(driver, "tables")


def test_reshape_tile_lds(driver):
    """No reshape tile asks for more than 64 KiB of LDS."""
    run(driver, "reshape")


def test_out_of_host_memory(driver):
    """Tables that do not fit in memory make an error, not an exception."""
    run(driver, "memory")


def test_stages(driver):
    """No length within a tile takes more stages than a launch holds."""
    run(driver, "stages")


def test_workgroups_of_few_lines(driver):
    """A pass over less than 20 KiB of points is not spread over workgroups."""
    run(driver, "few_lines")
