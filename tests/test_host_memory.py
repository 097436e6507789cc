"""Refused allocations in the host half of the library, on the CPU: tests/host_hip.cpp holds the scenarios and the
HIP runtime made of host memory that they run on."""
import os
import subprocess

import pytest

from ferrotensor_amd import build as ft_build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_hip")
    objs = []
    for src in (os.path.join(HERE, "host_hip.cpp"), os.path.join(ft_build.CSRC, "ft_runtime.cpp"),
                os.path.join(ft_build.CSRC, "ft_step.cpp")):
        obj = os.path.join(str(out), os.path.basename(src) + ".o")
        r = subprocess.run(["hipcc", "-x", "hip", "--cuda-host-only", *ft_build.FLAGS, "-O1", "-c", src, "-o", obj],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        objs.append(obj)
    exe = os.path.join(str(out), "host_hip")
    # kernels and their launchers are not linked: no scenario gets there
    r = subprocess.run(["g++", "-no-pie", "-Wl,--unresolved-symbols=ignore-all", *objs, "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("scenario", ["whole", "no_host_memory_for_the_list", "no_pinned_memory", "no_device_memory",
                                      "no_memory_for_another_rank"])
def test_host_half_with_refused_memory(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
