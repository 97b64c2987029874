"""The persistent kernels' claim loop on the CPU, with the kernels' own code
(tests/host/claim_emu.cpp), under the address and undefined-behaviour
sanitizers: 1 to 512 workgroups, both box grids, with and without copies of equal
tiles passed over, random tasks, group shapes and orders."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("claim") / "claim_emu")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(HERE, "host", "claim_emu.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("grid", [1, 7, 8, 64, 512])
def test_every_box_that_runs_is_claimed_once(emu, grid):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1")
    env.pop("LD_PRELOAD", None)
    for seed in range(6):
        for fold in "01":
            for mixed in "01":
                r = subprocess.run([emu, str(grid), fold, mixed, str(seed)], capture_output=True, text=True,
                                   env=env, timeout=60)
                assert r.returncode == 0 and "claim_emu: ok" in r.stdout, r.stdout + r.stderr
