"""One context whose runs change plan (smaller, larger, smaller again), precision
and task list, launched directly and as a replayed graph: each run's queues and
task energies pass through host memory that is kept between runs, so every
result has to be, bit for bit, that of a context used for it alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLANS = [([3], [5]), ([2, 3, 2], [4, 5, 2, 3]), ([1, 2], [3, 2])]


def _context(xt, ctx, plan, seed):
    O, V = sum(plan[0]), sum(plan[1])
    ctx.set_tiling(xt.Tiling(O, V, *plan), True)
    ctx.upload(xt.synth_closed_shell(O, V, seed, 0.05, 1e-2))
    print(f"[gpu] run buffers {plan} tasks={ctx.num_tasks()}", flush=True)


@pytest.mark.parametrize("graph", [0, 1])
def test_results_of_a_reused_context(xt, graph):
    kept = xt.CCSDTriples(0)
    for seed, plan in enumerate(PLANS):
        _context(xt, kept, plan, seed)
        n = kept.num_tasks()
        for prec in (xt.PREC_FP64, xt.PREC_MIXED):
            alone = xt.CCSDTriples(0)
            _context(xt, alone, plan, seed)
            want = alone.run(precision=prec)
            alone.close()
            for which in (None, [n - 1], None, list(range(n))[::-2]):
                if which is None:
                    got = kept.run(precision=prec, use_graph=graph)
                    assert (got["e4"], got["e5"]) == (want["e4"], want["e5"])
                    assert np.array_equal(got["task_partials"], want["task_partials"])
                else:
                    got = kept.run_tasks(which, precision=prec, use_graph=graph)
                    assert np.array_equal(got["task_partials"], want["task_partials"][which])
    kept.close()
