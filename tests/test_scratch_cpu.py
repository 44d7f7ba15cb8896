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


@pytest.mark.parametrize("case", ["retry", "idle", "sorted", "fitting", "trim"])
def test_scratch(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_device_array_reclaims(monkeypatch):
    """A DeviceArray that runs out of memory has the kept scratch freed first."""
    from abhsf_amd import hip

    class Runtime:
        free, error = 100, 0

        def hipMalloc(self, p, n):
            if n > self.free:
                self.error = 2
                return 2
            self.free -= n
            return 0

        def hipGetLastError(self):
            self.error = 0

        def hipFree(self, p):
            return 0

        def hipGetErrorString(self, rc):
            return b"out of memory"

    rt, calls = Runtime(), []

    def reclaim():
        calls.append(1)
        rt.free += 300
        return 300

    monkeypatch.setattr(hip, "_hip", rt)
    monkeypatch.setattr(hip, "reclaim", reclaim)
    hip.DeviceArray(40)
    assert calls == [1] and rt.error == 0
    with pytest.raises(hip.HipError):
        hip.DeviceArray(1000)
