"""The engine's host code on a fake HIP runtime (tests/engine_host): the built library is linked
behind it, so the decisions of lc2e_engine.cpp and of the kernels' launchers -- which memory a
launch uses, how a batch is split, what happens where memory runs out -- are the real ones, and
no GPU is needed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "engine_host")
LIB = os.path.join(ROOT, "lc2registration_amd", "_lib")


@pytest.fixture(scope="module")
def engine_test(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("a host C++ compiler and the HIP headers are needed")
    if not os.path.exists(os.path.join(LIB, "liblc2e.so")):
        from lc2registration_amd import build
        build.build()
    exe = str(tmp_path_factory.mktemp("engine_host") / "engine_test")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wextra", "-Wno-unused-parameter",
                    "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "lc2registration_amd", "csrc"),
                    os.path.join(HERE, "fake_hip.cpp"), os.path.join(HERE, "engine_test.cpp"),
                    "-o", exe, "-rdynamic", "-pthread", "-L" + LIB, "-llc2e", "-Wl,-rpath," + LIB,
                    "-Wl,--allow-shlib-undefined"], check=True, timeout=240)
    return exe


@pytest.mark.parametrize("scenario", [
    "noalloc_has_its_own_workspace",
    "noalloc_runs_in_large_parts",
    "captured_launches_keep_their_workspace",
    "a_refused_workspace_is_not_asked_for_again",
    "kept_memory_makes_room",
    "releases_leave_the_current_device",
    "every_device_gets_its_lds_limit",
    "launches_stay_below_the_runtime_limit",
    "noalloc_admits_what_it_did",
    "small_2d_launches_have_short_waves",
    "one_pose_of_a_stack_fills_the_device",
    "small_calls_have_few_commands",
    "small_3d_launches_are_spread_out",
    "chunks_fit_the_kernel_that_runs",
    "joint_histograms_that_warp_again_spread_out",
    "old_blocks_make_room_for_new_ones",
    "small_uploads_make_nothing_pinned",
    "a_pair_makes_two_pinned_blocks",
])
def test_engine_host(engine_test, scenario):
    r = subprocess.run([engine_test, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and f"{scenario} passed" in r.stdout, r.stdout + r.stderr
