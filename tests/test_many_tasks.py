"""Plans on both sides of the number of tasks from which only the queue entries
in use are brought and the task energies are converted by many workgroups
(kManyTasks, exachem_amd/csrc/xt_kernels.hip): whole runs, and subsets of one
task, of some in another order and of all but one, in both launch forms, give
the same task energies bit for bit, and totals that are their fixed-order sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLANS = {980: (3, 17), 1012: (1, 32), 1512: (3, 20), 4368: (5, 20)}


@pytest.mark.parametrize("n", list(PLANS))
def test_runs_of_plans_with_many_tasks(xt, oracle, n):
    O, V = PLANS[n]
    tiling = xt.Tiling.uniform(O, V, 2, 3)
    s = xt.synth_closed_shell(O, V, 11, 0.05, 1e-2)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(tiling, True)
    ctx.upload(s)
    assert ctx.num_tasks() == n
    print(f"[gpu] {n} tasks", flush=True)
    t = oracle.Tiling(tiling.occ, tiling.occ, tiling.vir, tiling.vir)
    e4, e5, ref = oracle.run_spatial(t, np.concatenate([s["eo"], s["eo"], s["ev"], s["ev"]]), s, True)
    rng = np.random.default_rng(2)
    some = rng.permutation(n)[:n // 3 | 1]
    for graph in (0, 1):
        r = ctx.run(use_graph=graph)
        p = r["task_partials"]
        if not graph:
            first = p
            assert np.all(np.abs(p - np.asarray(ref)) <= 1e-10 + 2e-14 * np.abs(ref))
        assert np.array_equal(p, first)
        assert (r["e4"], r["e5"]) == xt.sum_task_energies(p)
        for which in ([n - 1], some, [0], np.arange(n)[1:], rng.permutation(n)):
            q = ctx.run_tasks(which, use_graph=graph)
            assert np.array_equal(q["task_partials"], p[which])
            a = b = 0.0
            for x, y in p[which]:
                a, b = a + x, b + y
            assert (q["e4"], q["e5"]) == (a, b)
    ctx.close()
