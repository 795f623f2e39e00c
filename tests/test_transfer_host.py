"""copy_out (transfer.hip) without a GPU: its own source built with the host
compiler over plain-memory HIP calls that refuse pinned memory, events or
threads. A copy that cannot have its ring, or all of its threads, still
delivers. Sizes at the edges of its ranges; copies are exact."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIZES = ["524288", "2097151", "2097152", "16777215", "40000003"]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("needs g++ and the HIP headers")
    out = str(tmp_path_factory.mktemp("transfer") / "transfer_host")
    csrc = os.path.join(ROOT, "femeko.jl_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + csrc, "-x", "c++",
                    os.path.join(ROOT, "tests", "native", "transfer_host.cpp"), os.path.join(csrc, "transfer.hip"),
                    "-o", out, "-ldl", "-lpthread", "-rdynamic"], check=True)
    return out


@pytest.mark.parametrize("mode,way", [("all", "ring threads 7"), ("no_pinned", "plain threads 0"),
                                      ("no_event", "plain threads 0"), ("threads 0", "ring threads 0"),
                                      ("threads 1", "ring threads 1"), ("threads 4", "ring threads 4"),
                                      ("threads 6", "ring threads 6")])
def test_copies(program, mode, way):
    r = subprocess.run([program] + mode.split() + SIZES, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout.splitlines() == ["OK " + way] * len(SIZES)
