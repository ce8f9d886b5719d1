"""CPU: a session's memory (csrc/memory.h, memory.cpp) against a stand-in HIP
runtime that knows what is captured and what still runs."""
import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = tmp_path_factory.mktemp("memory") / "memory_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", f"-I{ROOT / 'tests/memory'}",
                    f"-I{ROOT / 'affon_amd/csrc'}", str(ROOT / "tests/memory/memory_test.cpp"),
                    str(ROOT / "affon_amd/csrc/memory.cpp"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("check", ["reuse", "other_stream", "capture", "capture_large", "no_free_in_capture",
                                   "no_idle_moment", "other_capture", "other_capture_scratch", "full", "exact_size",
                                   "scratch_between_threads", "host_memory_fails"])
def test_session_memory(driver, check):
    result = subprocess.run([str(driver), check], capture_output=True, text=True, timeout=60)
    assert result.returncode == 0, result.stdout + result.stderr
