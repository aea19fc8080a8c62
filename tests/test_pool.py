"""Device memory kept between trees (csrc/pool.hip): what is kept, for how long
and when it is given back, with a host allocator in the place of the device's;
and the sizes of a build's first list buffers."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "fmmgen_amd", "csrc")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    from fmmgen_amd.build import HIPCC
    d = tmp_path_factory.mktemp("pool")
    objs = []
    for src in (os.path.join(CSRC, "pool.hip"), os.path.join(HERE, "pool_harness.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-I", CSRC, "-c", src,
                        "-o", objs[-1]], check=True)
    exe = str(d / "pool_harness")
    subprocess.run(["g++", *objs, "-pthread", "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("check", ["scope_gives_back", "exact_size", "idle_gives_back", "bounded", "threads", "devices",
                                   "trim", "list_buffers"])
def test_pool(harness, check):
    r = subprocess.run([harness, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


def test_trim_without_kept_memory():
    import fmmgen_amd
    assert fmmgen_amd.trim_memory() == 0
