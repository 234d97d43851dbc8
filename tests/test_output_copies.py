"""How outputs reach the caller's arrays (csrc/host/Bert.cpp), on the CPU: tests/output_copies.cpp runs the host class over a
pretended device under AddressSanitizer + UndefinedBehaviorSanitizer."""
import os
import subprocess

import pytest

from test_host_sanitized import HERE, HOST, ROOT, _clang


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    clang = _clang()
    if clang is None:
        pytest.skip("no clang++ with sanitizer runtimes")
    exe = str(tmp_path_factory.mktemp("output_copies") / "output_copies")
    cmd = [clang, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
           "-mllvm", "-asan-globals=0", "-fno-omit-frame-pointer", "-I" + os.path.join(ROOT, "include"), "-I" + HOST,
           os.path.join(HERE, "output_copies.cpp"), os.path.join(HOST, "Bert.cpp"), "-o", exe]
    built = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if built.returncode != 0 and "sanitizer" in built.stdout.lower() and "not supported" in built.stdout.lower():
        pytest.skip("sanitizer runtimes not installed: " + built.stdout[-300:])
    assert built.returncode == 0, built.stdout[-3000:]
    return exe


# arrive: from less than a piece to several pieces and a remainder; throw: an output call that throws half-way leaves nothing that
# names its caller's arrays, which are freed before the next call; known: what is not ordinary host memory is left to the runtime's copy;
# lock: page-locked memory of some size only for a caller of large outputs, who is also served where there is none
@pytest.mark.parametrize("what", ["arrive", "throw", "known", "lock"])
def test_outputs(driver, what):
    run = subprocess.run([driver, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert run.returncode == 0 and "output_copies ok" in run.stdout, run.stdout[-4000:]
