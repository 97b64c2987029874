"""Boxes of equal tiles run once for all their antisymmetric copies
(fold_weight, exachem_amd/csrc/xt_queue.h)."""
import os
import shutil

import numpy as np
import pytest

from tests.test_gpu_parity import close, load_case, small_cases
from tests.test_host_safety import _build_and_run

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_weights_cover_every_box_once(tmp_path):
    r = _build_and_run(os.path.join(HERE, "host", "fold_check.cpp"), tmp_path)
    assert r.returncode == 0 and "fold_check: ok" in r.stdout, r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["uneven_small", "uneven_small_unrestricted"])
def test_integrals_without_the_exchange_symmetry_run_every_box(xt, oracle, name):
    """vvoo that misses (ai|bj) = (bj|ai) leaves the singles term without the
    antisymmetry the folding rests on: every box runs, and E[5] follows the
    oracle's sum over all elements of the unsymmetric array."""
    case = next(c for c in small_cases() if c["name"] == name)
    ctx, s = load_case(xt, case)
    rng = np.random.default_rng(3)
    s = dict(s, vvoo=s["vvoo"] + 0.02 * rng.normal(size=s["vvoo"].shape),
             t1=100.0 * s["t1"])
    print(f"[gpu] unsymmetric vvoo {name}", flush=True)
    ctx.upload(s)
    r = ctx.run()
    t = oracle.Tiling(case["occ_tiles"], case["occ_tiles"], case["vir_tiles"], case["vir_tiles"])
    evl = np.concatenate([s["eo"], s["eo"], s["ev"], s["ev"]])
    e4, e5, ref = oracle.run_spatial(t, evl, s, case["restricted"])
    assert close(r["e4"], e4) and close(r["e5"], e5), (r["e5"], e5)
    assert all(close(a, b) for a, b in zip(r["task_partials"].ravel(), ref.ravel()))
    ctx.close()
