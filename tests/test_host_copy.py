"""Host code on a stand-in for the HIP runtime (tests/host_copy/hip/hip_runtime.h).

Field and parameter reads (csrc/host_copy.cpp), where a chosen call can fail:
the values delivered, and what is left behind when a copy fails.  Batches
(csrc/batch.cpp) on runtimes of several versions: when steps replay a graph."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ehd-convection-3d_amd", "csrc")
HERE = os.path.join(ROOT, "tests", "host_copy")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not on PATH")


def _build(folder, harness, source):
    exe = str(folder / "harness")
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-g", "-Wall", "-I", HERE, os.path.join(HERE, harness),
                        os.path.join(CSRC, source), os.path.join(CSRC, "ehd_error.cpp"), "-o", exe, "-lpthread"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    exe = _build(tmp_path_factory.mktemp("host_copy"), "harness.cpp", "host_copy.cpp")

    def scenario(*args):
        r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
    return scenario


def test_small_and_large_reads_are_exact(run):
    run("exact")


@pytest.mark.parametrize("call", ["hipMemcpyAsync", "hipEventRecord", "hipEventSynchronize"])
def test_a_failed_copy_leaves_none_on_the_stream(run, call):
    run("failing", call)


def test_lack_of_host_memory_leaves_no_copy_on_the_stream(run):
    run("no_memory")


@pytest.mark.parametrize("call", ["hipHostMalloc", "hipEventCreateWithFlags"])
def test_reads_without_staging_memory_are_exact_and_leave_no_error(run, call):
    run("no_staging", call)


def test_a_stream_of_another_device_is_read(run):
    run("other_device")


@pytest.mark.parametrize("devices", [1, 3, 8, 9])
def test_staging_memory_is_kept_and_bounded(run, devices):
    run("kept", str(devices))


def test_a_read_leaves_nothing_to_its_streams_owner(run):
    run("waited")


@pytest.fixture(scope="module")
def batch_harness(tmp_path_factory):
    return _build(tmp_path_factory.mktemp("batch"), "batch_harness.cpp", "batch.cpp")


# 11 steps: the direct one, pairs of steady ones, and the last, which runs eagerly;
# two boxes of other planes, so the tuner captures a pair of each kind of step
@pytest.mark.parametrize("tune", [0, 2])
@pytest.mark.parametrize("version,replays", [(70200000, True), (70254321, True), (70051831, False), (60443483, False),
                                             (80000000, False)])
def test_batches_replay_graphs_only_on_the_runtime_they_were_built_for(batch_harness, version, replays, tune):
    for flags, graph in ((1 | tune, replays), (tune, False)):
        r = subprocess.run([batch_harness, str(version), str(flags)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        captures, played, launches = (int(w) for w in r.stdout.split()[::2])
        assert (captures > 0) == graph and played == (4 if graph else 0)
        # the tuner may keep one LBM launch for both boxes or one each
        assert graph or launches in (11, 22)
