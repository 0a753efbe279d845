"""LSParticle::finalize (fundem_amd/include/fundem/LSParticle.h) before the
bodies are on the device: a caller's arrays get the bodies as they were added
(orientations normalised), zero forces and torques. A host program, no GPU
call, in both storage precisions."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from fundem_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_bodies_as_added_before_initialize(precision, tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    core, _ = build.libs(precision)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if cxx is None or not os.path.exists(core) or not os.path.isdir(os.path.join(rocm, "include")):
        pytest.skip("no host compiler, core library or HIP headers")
    exe = tmp_path / "state_rows_check"
    lib = os.path.dirname(core)
    subprocess.run([cxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-Wno-unused-result",
                    *(["-DFDM_STATE_FP64"] if precision == "fp64" else []), "-I", os.path.join(rocm, "include"),
                    os.path.join(HERE, "state_rows_check.cpp"), "-o", str(exe), "-L", lib,
                    "-l" + os.path.basename(core)[3:-3], "-L", os.path.join(rocm, "lib"), "-lamdhip64",
                    "-Wl,-rpath," + lib, "-Wl,-rpath," + os.path.join(rocm, "lib"), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stderr)
    got = np.array([[float(c) for c in line.split()] for line in r.stdout.splitlines()])
    b = 10.0 * np.arange(5)[:, None]
    want = np.concatenate([b + [0.1, 0.2, 0.3], b + [1, 2, 3], b + [4, 5, 6], np.zeros((5, 6))], axis=1)
    assert got.shape == (5, 19) and np.array_equal(got[:, :15], want)
    assert np.abs(got[:, 15:] - [0.0, 0.0, 0.6, 0.8]).max() < 1e-15
