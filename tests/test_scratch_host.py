"""The scratch buffers of csrc/runtime.cpp, compiled for the CPU against a HIP runtime made of
counters (tests/native/scratch_host.cpp): threads, captures and failing allocations."""
import subprocess
from pathlib import Path

import pytest

from tilers_hip import _build

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("scratch") / "scratch_host"
    # the rest of runtime.cpp refers to HIP functions that no scenario reaches
    cmd = ["g++", "-O1", "-g", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__",
           "-I", str(_build.ROCM / "include"), "-I", str(_build.CSRC),
           str(ROOT / "tests" / "native" / "scratch_host.cpp"), str(_build.CSRC / "runtime.cpp"),
           "-Wl,--unresolved-symbols=ignore-all", "-o", str(exe)]
    out = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert out.returncode == 0, out.stdout
    return exe


@pytest.mark.parametrize("scenario", [
    "per_thread_own", "per_thread_bounded", "short_of_memory", "short_of_memory_optional",
    "refused_while_recording", "another_stream_recorded"])
def test_scratch(program, scenario):
    out = subprocess.run([str(program), scenario], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
