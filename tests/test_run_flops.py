"""Flops that a run computes (xt_run_flops): the elements of the boxes that are
not copies of another under the exchange of equal tiles, counted box by box."""
import itertools

import numpy as np
import pytest


def _elements(dims, tiles, prec):
    """(elements in boxes that run, all elements) of a task."""
    ran = 1
    for s in (0, 3):
        w = 8 if prec and s else 4
        ext = [[min(w, d - w * k) for k in range(-(-d // w))] for d in dims[s:s + 3]]
        same = [tiles[s] == tiles[s + 1], tiles[s + 1] == tiles[s + 2]]
        ran *= sum(ext[0][a] * ext[1][b] * ext[2][c]
                   for a, b, c in itertools.product(*[range(len(e)) for e in ext])
                   if (not same[0] or a <= b) and (not same[1] or b <= c))
    return ran, int(np.prod(dims))


def test_before_an_upload_every_box_counts(xt):
    ctx = xt.CCSDTriples(-1)
    ctx.set_tiling(xt.Tiling(7, 22, [3, 4], [5, 9, 8]))
    total, per, _ = ctx.flops()
    for prec in (0, 1):
        got, each = ctx.run_flops(prec)
        assert got == total and np.array_equal(each, per)
    with pytest.raises(xt.XtError):
        ctx.run_flops(2)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("occ,vir", [([9, 4], [17, 8]), ([13], [33]), ([1, 2, 5], [3, 9])])
def test_count_of_the_boxes_that_run(xt, occ, vir):
    O, V = sum(occ), sum(vir)
    s = xt.synth_closed_shell(O, V, 5, 0.05, 1e-3)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling(O, V, occ, vir), False)
    tasks, _ = ctx.task_list()
    _, per, _ = ctx.flops()
    tiles = np.array(occ * 2 + vir * 2)
    ctx.upload(s)
    for prec in (0, 1):
        total, got = ctx.run_flops(prec)
        want = [p * np.divide(*_elements(tiles[t].tolist(), t.tolist(), prec)) for p, t in zip(per, tasks)]
        assert np.allclose(got, want, rtol=1e-13, atol=0) and np.isclose(total, np.sum(want), rtol=1e-13)
        assert total < per.sum()
    rng = np.random.default_rng(1)
    ctx.upload(dict(s, vvoo=s["vvoo"] + 0.1 * rng.normal(size=s["vvoo"].shape)))  # no symmetry: every box
    assert np.array_equal(ctx.run_flops(1)[1], per)
    ctx.close()


@pytest.mark.gpu
def test_analytic_schedule_follows_what_runs(xt):
    """Largest first onto the least-loaded queue, by the flops that a run computes."""
    tiling = xt.Tiling.uneven(16, 64, (3, 8), (9, 24), seed=4)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(tiling)
    ctx.synth_upload(1)
    for prec in (0, 1):
        _, cost = ctx.run_flops(prec)
        lay = ctx.queue_layout(precision=prec, schedule=xt.SCHED_ANALYTIC)
        loads = []
        for q in range(8):
            c = cost[lay["qtask"][lay["qbeg"][q]:lay["qbeg"][q + 1]]]
            assert np.all(np.diff(c) <= 0)
            loads.append(c.sum())
        assert max(loads) - min(loads) <= cost.max()
    ctx.close()
