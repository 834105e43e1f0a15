"""The pinned slots between host arrays and the device (st_hostcopy.hip), built for the CPU
on a simulated runtime (tests/hostcopy), with the thread sanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("needs clang++")
    exe = str(tmp_path_factory.mktemp("ring") / "ring")
    src = os.path.join(HERE, "hostcopy")
    subprocess.run([CLANG, "-O1", "-g", "-std=c++17", "-Xarch_host", "-fsanitize=thread", "-I", src, os.path.join(src, "ring.cpp"),
                    "-o", exe, "-pthread"], check=True)
    return exe


def run(exe, *args):
    r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
    if "FATAL: ThreadSanitizer" in r.stderr:
        pytest.skip("the thread sanitizer does not start here")
    assert r.returncode == 0 and not r.stderr, r.stdout + r.stderr[:2000]


def test_arrays_of_all_sizes_arrive(ring):
    run(ring, "sizes")


def test_pinned_arrays_take_the_runtime_s_copy(ring):
    run(ring, "known")


@pytest.mark.parametrize("case", ["failed_out", "failed_in"])
@pytest.mark.parametrize("at", [1, 3, 12, 18])
def test_a_copy_may_fail_while_threads_copy(ring, case, at):
    run(ring, case, at)


@pytest.mark.parametrize("case", ["failed_out_then", "failed_in_then"])
@pytest.mark.parametrize("at", [1, 3, 12, 18])
def test_copies_after_a_failed_one_arrive(ring, case, at):
    """A transfer that was queued before the failure must not reach a slot, or leave one, once
    the next copy uses it."""
    run(ring, case, at)
