"""The helpers that move large outputs (csrc/host/CopyTeam.h), on the CPU: tests/copy_team.cpp under ThreadSanitizer, with all the
processors, two and one, and with a thread library that gives fewer threads than are asked for."""
import os
import subprocess

import pytest

from test_host_sanitized import HERE, HOST, _clang


def build(tmp_path, flags):
    clang = _clang()
    if clang is None:
        pytest.skip("no clang++")
    exe = str(tmp_path / "copy_team")
    cmd = [clang, "-std=c++17", "-O1", "-g", "-I" + HOST] + flags + [os.path.join(HERE, "copy_team.cpp"), "-o", exe, "-lpthread", "-ldl"]
    built = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if built.returncode != 0 and "tsan" in built.stdout.lower():
        pytest.skip("sanitizer runtime not installed: " + built.stdout[-300:])
    assert built.returncode == 0, built.stdout[-3000:]
    return exe


def run(exe, *args):
    done = subprocess.run([exe] + [str(a) for a in args], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    if "unexpected memory mapping" in done.stdout:
        pytest.skip("ThreadSanitizer does not start with this kernel's address layout")
    assert done.returncode == 0 and "copy_team ok" in done.stdout, done.stdout[-4000:]
    return done.stdout


@pytest.mark.parametrize("processors", [0, 2, 1])
def test_copies_under_thread_sanitizer(tmp_path, processors):
    run(build(tmp_path, ["-fsanitize=thread"]), processors)


@pytest.mark.parametrize("threads", [-1, 0, 1, 2, 4, 14])
def test_fewer_threads_than_asked_for(tmp_path, threads):
    """The first team takes what there is; those behind it have one helper, or none."""
    out = run(build(tmp_path, ["-DCOUNT_THREADS"]), 0, threads)
    started = int(out.split("threads ")[1].split()[0])
    assert started == threads or threads < 0


@pytest.mark.parametrize("processors", [1, 2, 3])
def test_no_more_helpers_than_other_processors(tmp_path, processors):
    """Eight teams, and three threads of the test's own."""
    if len(os.sched_getaffinity(0)) < processors:
        pytest.skip("fewer processors")
    assert "threads %d\n" % (3 + 8 * (processors - 1)) in run(build(tmp_path, ["-DCOUNT_THREADS"]), processors, -1)
