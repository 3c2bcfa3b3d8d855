"""csrc/resident_seat.h over a stand-in for the HIP runtime: how a resident kernel is launched, and which calls the launches of several models are surrounded by."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_INCLUDE = "/opt/rocm/include"


@pytest.fixture(scope="module")
def seats(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx or not os.path.exists(os.path.join(HIP_INCLUDE, "hip", "hip_runtime_api.h")):
        pytest.skip("no C++ compiler or HIP headers")
    exe = str(tmp_path_factory.mktemp("seat") / "check")
    csrc = os.path.join(ROOT, "forge-llm_amd", "csrc")
    r = subprocess.run([cxx, "-std=c++17", "-w", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", HIP_INCLUDE, "-I", os.path.join(ROOT, "include"), "-I", csrc,
                        os.path.join(ROOT, "tests", "resident_seat_check.cpp"), os.path.join(csrc, "resident_seat.cpp"), "-o", exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr

    def run(scenario, **env):
        out = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=60, env=dict(os.environ, **env))
        assert out.returncode == 0, out
        return out.stdout.split("\n")[:-1]
    return run


OK, HIP_ERROR = "-> 0", "-> -5"


def test_offsets_of_32_bits(seats):
    """A cache or an output matrix (Q8_0, Q4_0) of 4 GiB is left to the other kernels: the blocks behind would be read from its beginning."""
    assert seats("offsets") == ["1 0 1 0 1 0"]


def test_a_copy_for_speed_leaves_memory(seats):
    """The copy of a K-quant model's matrices is made where it takes an eighth of the free memory at most."""
    assert seats("copy") == ["1 0 0"]


@pytest.mark.parametrize("value,want", [("0", "ordinary"), ("1", "cooperative")])
def test_the_variable_asks_for_cooperative_launches(seats, value, want):
    assert seats("launch", FORGE_HIP_PD_COOP=value) == [f"{want} a 256 768 1000"]


def test_no_kernel_is_launched_past_it():
    """Both resident kernels go through resident_launch."""
    for name in ("decode_ahead.hip", "decode_persistent.hip"):
        with open(os.path.join(ROOT, "forge-llm_amd", "csrc", name)) as f:
            text = f.read()
        assert "resident_launch(" in text and "hipLaunchKernel(" not in text and "hipLaunchCooperativeKernel(" not in text, name


def test_a_model_alone_pays_for_nothing(seats):
    assert seats("one") == ["launch a", OK, "launch a", OK]


def test_launches_on_two_streams_follow_one_another(seats):
    assert seats("two") == ["sync device 0", "launch a", "record a", OK, "launch a", "record a", OK, "wait b", "launch b", "record b", OK, "wait a", "launch a", "record a", OK]


def test_devices_do_not_wait_for_one_another(seats):
    """An event belongs to a device and is recorded on that device's streams only."""
    assert seats("devices") == ["launch a", OK, "launch c", OK, "launch a", OK, "sync device 1", "launch c", "record c", OK, "launch a", OK, "wait d", "launch d", "record d", OK]


def test_a_step_that_was_launched_is_not_reported_as_failed(seats):
    """The device advances position and counts: an error behind the launch would let the caller feed the token again."""
    assert seats("record fails") == ["sync device 0", "launch a", "sync a", OK, "launch b", "record b", OK, "wait a", "launch a", "record a", OK]


def test_a_step_that_cannot_wait_is_not_launched(seats):
    assert seats("wait fails") == ["sync device 0", "launch a", "record a", OK, HIP_ERROR]
