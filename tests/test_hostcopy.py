"""The ring of pinned chunks behind large copies (m2c_hostcopy.h), on a
stand-in for the runtime: which memory goes through it, that every byte
arrives, that failures end in an error code and not in a wait, and (built with
ThreadSanitizer) that the threads' accesses to the ring are ordered."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MB = 1 << 20


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostpipe") / "driver")
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-fsanitize=thread",
                           "-I" + os.path.join(HERE, "hostpipe"), "-o", exe, os.path.join(HERE, "hostpipe", "driver.cpp")])

    def run(*args):
        r = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=60,
                           env=dict(os.environ, TSAN_OPTIONS="halt_on_error=1"))
        assert r.returncode == 0, r.stderr[-2000:]
        return [tuple(int(x) for x in line.split()) for line in r.stdout.split("\n") if line]

    return run


@pytest.mark.parametrize("way", ["up", "down"])
@pytest.mark.parametrize("what", ["pageable", "older-runtime"])
@pytest.mark.parametrize("n", [8 * MB, 8 * MB + 1, 16 * MB, 37 * MB + 123])
def test_pageable_memory_goes_through_the_ring(driver, way, what, n):
    assert driver(what, way, n) == [(0, 1, -(-n // (2 * MB)), 0)] * 2


@pytest.mark.parametrize("way", ["up", "down"])
@pytest.mark.parametrize("what,n", [("pinned", 40 * MB), ("pinned-head", 40 * MB), ("pinned-tail", 40 * MB),
                                    ("pageable", 8 * MB - 1), ("no-pinned-memory", 40 * MB)])
def test_other_memory_is_left_to_the_runtime(driver, way, what, n):
    """The link reads and writes pinned memory itself: staged, it would be
    copied once more by the CPU."""
    assert driver(what, way, n) == [(0, 1, 1, 1)] * 2


@pytest.mark.parametrize("way", ["up", "down"])
def test_a_failing_copy_is_reported(driver, way):
    first, second = driver("link-fails", way, 40 * MB)
    assert first[0] != 0 and first[2] == 5
    assert second[:3] == (0, 1, 20)


def test_solvers_share_a_ring(driver):
    """One after another they use the same one; it goes with the last of them."""
    assert driver("solvers", "up", 9 * MB, 5) == [(0, 1, 1, 0)]


def test_solvers_copying_at_once(driver):
    """Each copy has a ring to itself, and at most two are kept."""
    (bad, allocated, held, left), = driver("solvers", "down", 9 * MB, 5)
    assert bad == 0 and 1 <= allocated <= 15 and 1 <= held <= 2 and left == 0
