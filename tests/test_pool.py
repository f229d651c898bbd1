"""CPU check of the pool of kept device memory (qs_pool.hip): tests/cpp/
pool_check.cpp compiles that file against a stand-in for the HIP runtime and
runs its rules one by one."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pool") / "pool_check")
    subprocess.run(["g++", "-x", "c++", "-std=c++17", "-O1", "-pthread",
                    "-I", os.path.join(CPP, "fake_hip"),
                    "-I", os.path.join(ROOT, "quaru_amd", "csrc"),
                    os.path.join(CPP, "pool_check.cpp"), "-ldl", "-o", out],
                   check=True, capture_output=True, timeout=300)
    return out


@pytest.mark.parametrize("rule", ["bounds", "idle", "capture", "no_thread", "freeing", "device", "release"])
def test_kept_memory(exe, rule):
    res = subprocess.run([exe, rule], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout + res.stderr
