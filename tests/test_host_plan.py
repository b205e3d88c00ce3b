"""The tiled plan's host side (csrc/sloth_tiled.hip) compiled for the host with a
HIP runtime that records launches (tests/host_plan/plan_host.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    from sloth_amd import _build

    exe = str(tmp_path_factory.mktemp("plan") / "plan_host")
    subprocess.run([_build.hipcc(), "--offload-host-only", "-x", "hip", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"),
                    "-I", _build.CSRC, os.path.join(HERE, "host_plan", "plan_host.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["careful_room", "odd_reach"])
def test_plan(host, what):
    r = subprocess.run([host, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
