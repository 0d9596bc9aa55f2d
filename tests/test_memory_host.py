"""The library's host-side device-memory code (csrc/pool.cpp,
csrc/levels.hpp, csrc/pack.cpp) on the CPU, over
a fake device, under AddressSanitizer and UndefinedBehaviorSanitizer."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("needs g++ and the HIP headers")
    out = tmp_path_factory.mktemp("memory")
    subprocess.run(["make", "-s", "-C", os.path.join(HERE, "sanitize"), f"OUT={out}", f"ROCM={ROCM}",
                    f"{out}/memory_driver"], check=True, capture_output=True, timeout=600)
    return str(out / "memory_driver")


def run(driver, check, want):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:exitcode=3", OMP_NUM_THREADS="2")
    r = subprocess.run([driver, check], capture_output=True, text=True, env=env, timeout=120)
    assert r.returncode == 0 and r.stdout.split("\n")[:len(want)] == want, r.stdout[-2000:] + r.stderr[-4000:]
    assert "runtime error" not in r.stderr and "AddressSanitizer" not in r.stderr, r.stderr[-4000:]


def test_memory_given_back_while_the_process_ends(driver):
    run(driver, "end_of_process", ["end_of_process ok", "late ok"])


def test_allocation_that_fails_while_another_thread_flushes(driver):
    run(driver, "flushed_by_another", ["flushed_by_another ok"])


def test_what_index_builds_take_of_little_memory(driver):
    run(driver, "index_builds", ["index_builds ok"])


def test_blocks_freed_while_a_stream_records(driver):
    run(driver, "given_while_capturing", ["given_while_capturing ok"])


def test_level_buffers_when_memory_runs_out(driver):
    run(driver, "growth_that_fails", ["growth_that_fails ok"])


def test_network_buffers_when_memory_runs_out(driver):
    run(driver, "network_that_does_not_fit", ["network_that_does_not_fit ok"])


def test_kept_memory_with_several_threads_and_given_back(driver):
    run(driver, "threads", ["threads ok"])


@pytest.mark.gpu
def test_trim():
    """The index of a released graph stays with the library until it is asked
    for; the counts of later graphs do not depend on it."""
    import cuts_amd as F
    ctx = F.Context()
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime that the library has loaded

    def free_bytes():
        fr, tot = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(fr), ctypes.byref(tot)) == 0
        return fr.value

    ctx.trim()
    g = F.Graph.chung_lu(20000, 100000, 2.2, 900, 3)
    p = F.Plan(F.Graph.from_edges(4, [(0, 1), (1, 2), (2, 0), (2, 3)]))
    dg = ctx.upload(g)
    want = ctx.match(dg, p).count
    del dg
    before = free_bytes()
    freed = ctx.trim()
    assert freed >= 1 << 20
    assert free_bytes() - before >= freed // 2
    assert ctx.trim() == 0
    assert ctx.match(ctx.upload(g), p).count == want
