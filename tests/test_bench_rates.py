"""bench.py's roofline counts the flops that a launch computes."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_roofline_counts_the_boxes_that_run(xt, prec):
    print(f"[gpu] bench O=8 V=48 {prec}", flush=True)
    r = subprocess.run(
        [sys.executable, os.path.join(ROOT, "bench.py"), "--config", "c0", "--precision", prec, "--steps", "2",
         "--warmup", "1", "--no-cpu-baseline", "--no-compare", "--no-physical", "--gather-tasks", "0",
         "--dropin-tasks", "0", "--cholesky-leg", "0", "--budget-s", "60"],
        capture_output=True, text=True, timeout=110, cwd=ROOT)
    assert r.returncode == 0, r.stderr[-2000:]
    line = json.loads(r.stdout.strip().splitlines()[-1])
    roof, ms = line["roofline"], line["roofline"]["kernel_ms"]
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling.uniform(8, 48, 8, 16))
    total, _, parts = ctx.flops()
    ctx.synth_upload(1)
    ran, _ = ctx.run_flops(xt.PREC_MIXED if prec == "mixed" else xt.PREC_FP64)
    ctx.close()
    assert ran < total and roof["flops_per_launch"] == ran
    assert abs(roof["achieved"] - ran / ms / 1e9) <= 1e-9 * roof["achieved"] and roof["frac"] < 1
    assert abs(line["tflops"] - total / ms / 1e9) <= 1e-9 * line["tflops"]
    if prec == "mixed":
        assert roof["mfma_issued_tflops"] <= 3 * ran / ms / 1e9
