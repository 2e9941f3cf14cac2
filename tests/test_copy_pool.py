"""CPU test of the threads that empty staging slots (csrc/copy_pool.h): every
byte arrives for any number of chunks and threads, a copy can be given up, and
threads that wait for a stream's work sleep instead of spinning through it."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "lowlevelfem.jl_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("pool") / "copy_pool_check"
    r = subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", os.path.join(ROOT, "tests", "copy_pool_check.cpp"),
                        "-o", str(exe), "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return lambda *a: subprocess.run([str(exe), *map(str, a)], capture_output=True, text=True, timeout=60)


# one chunk, a full ring of eight, one more, remainders of a byte; slices of less than a cache line
@pytest.mark.parametrize("bytes_,chunk", [(1, 64), (100, 64), (4096, 512), (4097, 512), (3_000_001, 200_000)])
@pytest.mark.parametrize("use", [1, 3, 8, 99])
def test_every_byte_arrives(check, bytes_, chunk, use):
    r = check("copy", bytes_, chunk, use)
    assert r.returncode == 0 and r.stdout.strip() == "1"


def test_given_up(check):
    r = check("abandon")
    assert r.returncode == 0 and r.stdout.strip() == "1"


# Eight threads that spin through two waits of 300 ms take 0.6 s of CPU time
# each, as far as there are processors; asleep they take 0.2 ms a wait.
def test_threads_sleep_while_nothing_comes(check):
    r = check("idle", 300)
    assert r.returncode == 0 and float(r.stdout) < 100.0
