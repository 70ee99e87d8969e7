"""The host runtime (h-blast_amd/csrc/hb_seed.cpp, hb_batch.cpp, hb_serve.cpp)
on the CPU, over a stand-in for the HIP runtime and the kernels
(tests/hostrt): what it does with memory, errors and streams when a call
fails.  Kernels and results are the GPU tests' matter."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "h-blast_amd", "csrc")
HERE = os.path.join(ROOT, "tests", "hostrt")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SRC = [os.path.join(CSRC, f) for f in ("hb_seed.cpp", "hb_batch.cpp", "hb_serve.cpp", "hb_seq.cpp",
                                       "hb_hdb.cpp", "hb_balance.cpp", "hb_seg.cpp",
                                       "hb_cosched.cpp")]
SRC += [os.path.join(HERE, f) for f in ("fake_hip.cpp", "driver.cpp")]

pytestmark = pytest.mark.skipif(
    shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip")),
    reason="g++ or the HIP headers not installed")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("hostrt")
    flags = ["-O1", "-g", "-std=c++17", "-w", "-pthread", "-fsanitize=address,undefined",
             "-fno-sanitize-recover=all", "-D__HIP_PLATFORM_AMD__",
             "-include", os.path.join(HERE, "fake_hip.h"), "-I" + os.path.join(ROCM, "include"),
             "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-I" + HERE]
    jobs = []
    for s in SRC:
        o = str(tmp / (os.path.basename(s) + ".o"))
        jobs.append((o, subprocess.Popen(["g++", *flags, "-c", s, "-o", o])))
    for _, j in jobs:
        assert j.wait() == 0
    exe = str(tmp / "driver")
    subprocess.run(["g++", "-pthread", "-fsanitize=address,undefined", *[o for o, _ in jobs],
                    "-o", exe], check=True)
    return exe


def run(driver, name):
    r = subprocess.run([driver, name], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0:verify_asan_link_order=0"))
    assert r.returncode == 0, r.stderr[-4000:]


def test_failed_pass_leaves_no_results(driver):
    run(driver, "failed_collect")


def test_failed_call_waits_for_its_work(driver):
    run(driver, "failed_calls_wait")


def test_handled_errors_are_cleared(driver):
    run(driver, "handled_errors")


def test_pool_keeps_buffer_sizes(driver):
    run(driver, "pool_sizes")


def test_freed_databases_are_free_memory(driver):
    run(driver, "freed_memory")


def test_small_requests_leave_large_pinned_buffers(driver):
    run(driver, "pinned_buffers")


def test_uploads_from_memory_the_runtime_knows(driver):
    run(driver, "upload_sources")


def test_served_batches_order_within_the_budget(driver):
    run(driver, "served_order")


def test_database_outlives_its_context(driver):
    run(driver, "database_after_context")


def test_order_on_the_host(driver):
    run(driver, "host_order")
