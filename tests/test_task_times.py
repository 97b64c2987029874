"""Per-task device times: what the GPU spent, also where boxes of equal tiles
stand for their copies."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("occ,vir", [([12], [20]), ([9, 5], [17, 24])])
def test_task_times_fit_the_kernel_time(xt, occ, vir, prec):
    """One workgroup runs every box in turn, so the tasks' times add up to no
    more than the kernel's own (2% and 0.05 ms for the two clocks), and to most
    of it: what lies between boxes is a claim (30% allowed)."""
    O, V = sum(occ), sum(vir)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling(O, V, occ, vir), True)
    ctx.upload(xt.synth_closed_shell(O, V, 5, 0.05, 1e-3))
    print(f"[gpu] task times {occ} {vir} precision {prec}", flush=True)
    ctx.prepare(prec)
    r = ctx.run(precision=prec, record_task_time=1, workgroups=1)
    total = float(np.sum(r["task_ms"], dtype=np.float64))
    assert 0.7 * r["kernel_ms"] - 0.05 <= total <= 1.02 * r["kernel_ms"] + 0.05, (total, r["kernel_ms"])
    ctx.close()


def test_features_tell_the_tasks_that_run_in_part(xt):
    """Extents are negative exactly where a position is on the tile of the one
    before it, once integrals are uploaded that let copies be skipped."""
    occ, vir = [4, 4], [9, 9]
    s = xt.synth_closed_shell(8, 18, 5, 0.05, 1e-3)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling(8, 18, occ, vir), False)
    tasks, _ = ctx.task_list()
    tiles = np.array(occ * 2 + vir * 2)
    plain = tiles[tasks].astype(np.float32) / np.float32(48)
    sign = np.ones_like(plain)
    for a, b in ((0, 1), (1, 2), (3, 4), (4, 5)):
        sign[tasks[:, a] == tasks[:, b], b] = -1
    assert (sign < 0).any() and np.array_equal(ctx.task_features(1)[:, :6], plain)
    ctx.upload(s)
    assert np.array_equal(ctx.task_features(1)[:, :6], sign * plain)
    rng = np.random.default_rng(1)
    ctx.upload(dict(s, vvoo=s["vvoo"] + 0.1 * rng.normal(size=s["vvoo"].shape)))
    assert np.array_equal(ctx.task_features(1)[:, :6], plain)
    ctx.close()
