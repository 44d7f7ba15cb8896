"""The device scratch kept between operations (Arena, DevBuf in prims.hip),
run on the host against a stand-in for the HIP runtime with a memory limit."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("scratch") / "scratch_host")
    csrc = os.path.join(ROOT, "abhsf_amd", "csrc")
    objs = []
    for src in (os.path.join(csrc, "prims.hip"), os.path.join(ROOT, "tests", "native", "scratch_host.cpp")):
        objs.append(f"{out}.{len(objs)}.o")
        subprocess.check_call([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-I", csrc, "-c", src,
                               "-o", objs[-1]])
    # (the kernels' code object is left out: nothing is launched)
    subprocess.check_call(["g++", *objs, "-o", out, "-no-pie", "-pthread", "-Wl,--unresolved-symbols=ignore-in-object-files"])
    return out


@pytest.mark.parametrize("case", ["retry", "idle", "sorted", "fitting"])
def test_scratch(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
