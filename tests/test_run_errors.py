"""A run that fails part-way leaves nothing in flight on the context's stream
(tests/host/run_errors.cpp, over a stand-in for the HIP runtime; no GPU)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "exachem_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_failed_runs_leave_nothing_in_flight(tmp_path):
    srcs = [os.path.join(CSRC, "xt_host.cpp"), os.path.join(CSRC, "xt_gather.cpp"),
            os.path.join(HERE, "host", "run_errors.cpp")]
    objs = []
    for s in srcs:
        objs.append(str(tmp_path / (os.path.basename(s) + ".o")))
        subprocess.run([HIPCC, "-O1", "-std=c++17", "-fPIC", "--offload-host-only", "-c", s, "-o", objs[-1]],
                       check=True, capture_output=True)
    exe = str(tmp_path / "run_errors")
    subprocess.run(["g++", *objs, "-lpthread", "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "run_errors: ok" in r.stdout, r.stdout + r.stderr
