"""The pinned pool and the transfers' host side (csrc/sloth_stage.hip), compiled
with a HIP runtime of host memory (tests/host_stage/stage_host.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("stage") / "stage_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", "/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "rust-sloth_amd", "csrc"),
                    os.path.join(HERE, "host_stage", "stage_host.cpp"), "-o", exe], check=True)
    return exe


def _run(host, what):
    r = subprocess.run([host, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("what", ["small_lease", "pool_bound"])
def test_pinned_pool(host, what):
    _run(host, what)


@pytest.mark.parametrize("what", ["waits_asleep", "waits_asleep_long"])
def test_read_back_waits_asleep(host, what):
    _run(host, what)
