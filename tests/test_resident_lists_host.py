"""The lists of the resident launches on the SELL copy (resident_lists.h) built
and run on the host: every entry's column and every block's halo against their
definition (integers, equal), with threads or memory refused."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    out = str(tmp_path_factory.mktemp("lists") / "lists")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-I" + os.path.join(ROOT, "femeko.jl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "resident_lists_host.cpp"), "-o", out, "-ldl", "-lpthread",
                    "-rdynamic"], check=True)
    return out


def _run(program, *args):
    r = subprocess.run([program] + [str(a) for a in args], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout.split()


# one row; a block's edge and one row more; a short last slice; many blocks
@pytest.mark.parametrize("nv", [1, 511, 512, 513, 1030, 6000])
@pytest.mark.parametrize("R", [512, 1024, 2048])
def test_lists(program, nv, R):
    assert _run(program, nv, R, nv, 100, 100)[0] == "OK"


@pytest.mark.parametrize("threads", [0, 1, 5])
def test_fewer_threads(program, threads):
    assert _run(program, 6000, 512, 3, threads, 100) == _run(program, 6000, 512, 3, 100, 100)


# the working array of the caller's part, or of a thread's, cannot be had
@pytest.mark.parametrize("threads,arrays", [(0, 0), (100, 0), (100, 1)])
def test_no_memory(program, threads, arrays):
    assert _run(program, 6000, 512, 3, threads, arrays) == ["REFUSED"]
