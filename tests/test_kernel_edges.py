"""Both triples kernels and the per-task kernel at the edges of their boxes and
of their K chunks, against the CPU oracle: tile extents 1 to 9 (partial 4^6 and
4^3 x 8^3 boxes, every count of 16-row matrix tiles a side), contraction runs of
one to six units of 8, K tiles of the packed blocks around the chunk of 16.
Tolerances as in test_gpu_parity (stated there)."""
import numpy as np
import pytest

from tests.test_gpu_parity import MIX_TASK_FLOOR, MIX_TASK_REL, close, close_mixed

pytestmark = pytest.mark.gpu

SHAPES = [
    (3, 5, [1, 2], [2, 3]),
    (5, 9, [5], [4, 5]),
    (7, 8, [4, 3], [8]),
    (8, 17, [3, 5], [1, 9, 7]),
    (9, 16, [2, 4, 3], [16]),
    (9, 25, [4, 5], [9, 15, 1]),
    (17, 8, [8, 1, 8], [3, 5]),
    (12, 33, [6, 6], [17, 16]),
]


def _setup(xt, shape, seed):
    O, V, occ, vir = shape
    s = xt.synth_closed_shell(O, V, seed, 0.05, 1e-2)
    print(f"[gpu] edges O={O} V={V} {occ} {vir}", flush=True)
    return s, np.concatenate([s["eo"], s["eo"], s["ev"], s["ev"]])


@pytest.mark.parametrize("shape", SHAPES)
def test_kernels_at_box_and_chunk_edges(xt, oracle, shape):
    O, V, occ, vir = shape
    s, evl = _setup(xt, shape, 31)
    e4, e5, ref = oracle.run_spatial(oracle.Tiling(occ, occ, vir, vir), evl, s, True)
    ref = np.asarray(ref)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling(O, V, occ, vir), True)
    ctx.upload(s)
    r = ctx.run(precision=xt.PREC_FP64)
    assert close(r["e4"], e4) and close(r["e5"], e5), (r["e4"], e4, r["e5"], e5)
    assert all(close(a, b) for a, b in zip(r["task_partials"].ravel(), ref.ravel()))
    m = ctx.run(precision=xt.PREC_MIXED)
    floor = MIX_TASK_FLOOR * np.max(np.abs(ref[:, 0]))
    for got, want in zip(m["task_partials"], ref):
        assert np.all(np.abs(got - want) <= MIX_TASK_REL * abs(want[0]) + floor), (got, want)
    assert close_mixed(m["e4"], e4, e4, MIX_TASK_REL) and close_mixed(m["e5"], e5, e4, MIX_TASK_REL)
    ctx.close()


@pytest.mark.parametrize("shape", [SHAPES[k] for k in (0, 3, 5, 6, 7)])
def test_packed_kernel_at_k_tile_edges(xt, oracle, shape):
    from exachem_amd.hipmem import DevBuf, Stream
    O, V, occ, vir = shape
    s, evl = _setup(xt, shape, 32)
    t = oracle.Tiling(occ, occ, vir, vir)
    ref = np.asarray(oracle.run_spatial(t, evl, s, True)[2])
    so = oracle.expand_closed_shell(O, V, s["t1"], s["t2"], s["vvoo"], s["ovoo"], s["vvvo"])
    tasks, fac = oracle.task_list(t, True)
    offs = np.concatenate([[0], np.cumsum(t.tiles)])
    st = Stream()
    names = ("d1_t2", "d1_v2", "d2_t2", "d2_v2", "s1_t1", "s1_v2")
    for k in np.unique(np.linspace(0, len(tasks) - 1, 6).astype(int)):
        bufs, meta, _, sz = oracle.task_packed(t, so, tasks[k], True)
        dev = {n: DevBuf.from_array(bufs[n]) for n in names}
        dims = [int(t.tiles[b]) for b in tasks[k]]
        ev = [DevBuf.from_array(evl[offs[b]:offs[b] + t.tiles[b]]) for b in tasks[k]]
        nb = int(np.prod([(d + 3) // 4 for d in dims]))
        part = DevBuf(16 * nb)
        most = {n: sz[n] // (9 if n.startswith("s1") else sz["max_" + n[:2]]) for n in names}
        xt.fully_fused_ccsd_t_gpu(st.h, nb, dims, [dev[n].ptr for n in names], meta, t.noab, t.nvab,
                                  most, [e.ptr for e in ev], part.ptr)
        st.sync()
        p = part.to_array(2 * nb)
        got = fac[k] * np.sum(p[:nb]), fac[k] * np.sum(p[nb:])
        assert close(got[0], ref[k, 0]) and close(got[1], ref[k, 1]), (k, dims, got, ref[k])
        for b in list(dev.values()) + ev + [part]:
            b.free()
    st.destroy()
