"""The host side of the library: its launches over streams and events, and what it does when a runtime call or an allocation
fails.  Nothing runs on a GPU: the library is loaded onto a stand-in for the HIP runtime (fake_hip.cpp) in a process of its
own (host_pipeline.py)."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if not shutil.which("g++"):
        pytest.skip("no C++ compiler")
    out = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    os.path.join(HERE, "fake_hip.cpp"), "-o", out], check=True)
    return out


def run_check(fake_hip, check):
    r = subprocess.run([sys.executable, os.path.join(HERE, "host_pipeline.py"), fake_hip, check], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok"), r.stdout[-4000:]


@pytest.mark.parametrize("check", ["recovery-direct", "recovery-overlap", "recovery-timed", "clear-failed-direct", "clear-failed-overlap",
                                   "capture-direct", "capture-overlap", "capture-in-flight", "in-flight", "own-graph"])
def test_failed_calls_leave_the_cell_tables_empty(fake_hip, check):
    run_check(fake_hip, check)


def test_a_pipeline_does_without_the_kept_tables_where_memory_is_short(fake_hip):
    run_check(fake_hip, "short-memory")


def test_layers_with_few_channels_run_on_the_matrix_cores_in_large_tensors(fake_hip):
    run_check(fake_hip, "row-limits")


def test_strided_fp32_layers_with_16_channels_multiply_pairs(fake_hip):
    run_check(fake_hip, "strided-few-channels")


def test_layers_with_weights_that_are_not_finite_multiply_no_absent_neighbours(fake_hip):
    run_check(fake_hip, "weights-not-finite")


def test_configuring_a_layer_for_fp16_packs_its_weights_and_no_more(fake_hip):
    run_check(fake_hip, "first-configure")


def test_host_memory_that_runs_out_in_a_frame_is_an_error_code(fake_hip):
    run_check(fake_hip, "host-memory")


def test_every_event_of_an_overlapped_frame_is_waited_for(fake_hip):
    run_check(fake_hip, "events")


def test_layers_of_a_deep_backbone_do_not_wait_for_the_whole_coordinate_branch(fake_hip):
    run_check(fake_hip, "waits")


def test_small_frames_wait_for_a_pass_more_only_where_launches_are_shared(fake_hip):
    run_check(fake_hip, "own-waits")


def test_the_longer_branch_of_a_small_frame_is_launched_first(fake_hip):
    run_check(fake_hip, "order")


def test_first_layers_share_the_launches_of_coordinate_passes(fake_hip):
    run_check(fake_hip, "shared-launches")
