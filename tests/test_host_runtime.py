"""The library's host logic without a GPU: its calls go to a stand-in for the HIP runtime that hands out
addresses from a budget and notes launches, copies and waits (hip_stub.hpp)."""
import os
import subprocess

import pytest

import stwo_hip as S

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def memory_limit(tmp_path_factory):
    if not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("HIP headers not found")
    out = str(tmp_path_factory.mktemp("limit") / "memory_limit_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    os.path.join(HERE, "memory_limit_check.cpp"), "-o", out, "-rdynamic", "-ldl"], check=True,
                   capture_output=True)

    def run(case, kib):
        r = subprocess.run([out, S.LIB_PATH, case, str(kib)], capture_output=True, text=True, check=True)
        words = r.stdout.split()
        return {k: int(v) for k, v in zip(words[::2], words[1::2])}

    return run


@pytest.fixture(scope="module")
def downloads(tmp_path_factory):
    hipcc = os.environ.get("HIPCC", os.path.join(ROCM, "bin", "hipcc"))
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("download") / "download_check")
    subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"),
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    os.path.join(HERE, "download_check.cpp"), "-o", out], check=True, capture_output=True)
    return subprocess.run([out], capture_output=True, text=True, check=True).stdout.splitlines()


@pytest.mark.parametrize("stream", [0, 1], ids=["library stream", "another current stream"])
def test_copies_are_complete_on_return(downloads, stream):
    """Small and large copies to host memory, one on the device, one of odd length: each is enqueued on the
    current stream, and that stream is waited for."""
    assert downloads[stream].split() == ["11"] * 4


def test_copy_of_nothing_waits(downloads):
    assert downloads[2] == "1"


MIB = 1024


@pytest.mark.parametrize("case", ["lde", "plan"])
def test_extension_without_memory_for_matrices(memory_limit, case):
    """64 columns of 2^20 extended to 2^21: 53 MB of matrices make it faster.  Where they do not fit, the
    call runs on butterflies as it did before there were any."""
    assert memory_limit(case, 1000 * MIB) == {"status": 0, "matrices": 1, "butterflies": 0}
    assert memory_limit(case, 40 * MIB) == {"status": 0, "matrices": 0, "butterflies": 1}


def test_tuned_plan_without_memory_for_matrices(memory_limit):
    """The autotuner passes over a schedule whose matrices do not fit."""
    assert memory_limit("plan_tuned", 40 * MIB) == {"status": 0, "matrices": 0, "butterflies": 1}


@pytest.mark.parametrize("case,tables", [("interpolate", 1), ("evaluate", 2)])
def test_small_columns_without_memory_for_matrices(memory_limit, case, tables):
    """20000 columns of 2^12: a pointer table takes 157 KiB, the matrices 68.  The tables come first."""
    assert memory_limit(case, 157 * tables + 80) == {"status": 0, "matrices": 1, "butterflies": 0}
    assert memory_limit(case, 157 * tables + 10) == {"status": 0, "matrices": 0, "butterflies": 1}
    assert memory_limit(case, 150 * tables)["status"] != 0
