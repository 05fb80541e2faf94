"""The prompt path's host side on the CPU: prefill_host_driver.cpp defines the
HIP calls the library makes and lets chosen ones fail."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = "/opt/rocm"


@pytest.fixture(scope="module")
def seen(tmp_path_factory):
    """{observation: [value of the wide path, of batched steps]}"""
    exe = str(tmp_path_factory.mktemp("host") / "driver")
    lib = os.path.join(ROOT, "jetson-inference_amd")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-rdynamic",
                    "-I", os.path.join(ROOT, "include"), "-I", ROCM + "/include",
                    os.path.join(ROOT, "tests", "prefill_host_driver.cpp"), "-o", exe,
                    "-L", lib, "-l:libjinf_hip.so", "-L", ROCM + "/lib", "-lamdhip64",
                    f"-Wl,-rpath,{lib}:{ROCM}/lib"], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout
    got = {}
    for line in out.splitlines():
        k, v = line.split()
        got.setdefault(k, []).append(int(v))
    assert not any(got["engine"] + got["batch"] + got["first"])
    return got


def test_failed_prompt_leaves_the_sequence_where_it_was(seen):
    """The device position is written by a prompt's last chunk only, so a
    prompt that fails before it leaves the host's position alone too, and the
    next call goes on from there."""
    assert all(v != 0 for v in seen["failed"])
    assert seen["n_past"] == [5, 5]
    assert seen["again"] == [0, 0] and seen["from"] == [5, 5]
    assert seen["n_past_after"] == [8, 8]


def test_prompt_allocates_in_relaxed_capture_mode(seen):
    """The first wide prompt allocates its buffers: in the thread's relaxed
    capture mode, so that another thread's capture of the global mode neither
    refuses nor loses by it, and the thread's own mode is kept."""
    assert seen["allocs"][0] == 2 and seen["strict_allocs"] == [0, 0]
    assert seen["mode_kept"] == [1, 1]


def test_which_prompts_run_wide(seen):
    """8, 9, 16 and 17 tokens at 8 sequences and 65 at 64: more than one
    batched step runs wide, with large Q4_0 layers more than two steps of up
    to 32 rows."""
    assert seen["wide"] == [0, 1, 1, 1, 1] + [0, 0, 0, 1, 1] + [0, 1, 1, 1, 1]
