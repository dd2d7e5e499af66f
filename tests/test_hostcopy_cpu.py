"""The staged host transfers (hostcopy.cpp) compiled against a stand-in
runtime that runs every copy as late as the waits allow: bytes at the sizes
where the path changes, and each way a transfer can go short or fail."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostcopy") / "check")
    tests = os.path.join(ROOT, "tests")
    subprocess.run(["g++", "-O2", "-std=c++17", "-rdynamic", "-pthread", "-I", os.path.join(tests, "hip_stub"),
                    os.path.join(tests, "hostcopy_check.cpp"),
                    os.path.join(ROOT, "critic2_amd", "csrc", "hostcopy.cpp"), "-o", exe, "-ldl"], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)

    return run


def test_bytes(check):
    check("sizes")


@pytest.mark.parametrize("slots", [0, 1, 3])
def test_pinned_memory_runs_out(check, slots):
    """Fewer slots carry the transfer; with none the runtime's own pageable
    copy does, and files go through ordinary memory."""
    check("pinned", slots)


@pytest.mark.parametrize("threads", [0, 1, 3])
def test_threads_run_out(check, threads):
    check("threads", threads)


def test_a_file_that_ends_early(check):
    check("short")


def test_null_pointers(check):
    """An error of the runtime, whatever the size; nothing is read or written."""
    check("null")


def test_a_full_disk(check):
    check("full")


@pytest.mark.parametrize("copies", [0, 4])
@pytest.mark.parametrize("how", ["hip", "throw"])
def test_a_copy_that_fails(check, how, copies):
    """The first error comes out as the call's status with its message, no
    thread is left, and the context goes on working."""
    check(how, copies)


def test_two_contexts_at_once(check):
    check("two")


def test_batch_workers_share_the_slots(check):
    """However many workers, one context's slots and threads."""
    check("shared")
