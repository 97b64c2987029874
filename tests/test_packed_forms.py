"""Both forms of the per-task kernel's K chunks (packed_ends,
exachem_amd/csrc/xt_host.cpp): K tiles of 1 to 33 around the chunk of 16, several in
one chunk, one over several, a family of one tile, and the line between the
forms; both entry points, against the CPU oracle and each other bit for bit.
Tolerance as in test_gpu_parity (stated there)."""
import numpy as np
import pytest

from tests.test_gpu_parity import close

pytestmark = pytest.mark.gpu

SHAPES = [  # chunks with one per K tile / with tiles end to end, of one spin
    (6, 10, [1, 1, 1, 1, 2], [1, 2, 3, 1, 3]),  # 10 / 2
    (9, 34, [9], [17, 17]),                     # 5 / 4
    (8, 35, [3, 5], [16, 15, 4]),               # 5 / 4
    (17, 6, [1, 16], [6]),                      # 3 / 3
    (7, 33, [7], [33]),                         # 4 / 4
    (22, 22, [11, 11], [11, 11]),               # 4 / 4
    (5, 36, [5], [12, 12, 12]),                 # 4 / 4
    (33, 5, [8, 8, 8, 8, 1], [5]),              # 6 / 4
]


@pytest.mark.parametrize("shape", SHAPES)
def test_forms_match_the_oracle(xt, oracle, shape):
    from exachem_amd.hipmem import DevBuf, Stream
    O, V, occ, vir = shape
    s = xt.synth_closed_shell(O, V, 33, 0.05, 1e-2)
    evl = np.concatenate([s["eo"], s["eo"], s["ev"], s["ev"]])
    t = oracle.Tiling(occ, occ, vir, vir)
    so = oracle.expand_closed_shell(O, V, s["t1"], s["t2"], s["vvoo"], s["ovoo"], s["vvvo"])
    tasks, fac = oracle.task_list(t, False)
    ref = np.asarray(oracle.run_spatial(t, evl, s, False)[2])
    offs = np.concatenate([[0], np.cumsum(t.tiles)])
    st = Stream()
    names = ("d1_t2", "d1_v2", "d2_t2", "d2_v2", "s1_t1", "s1_v2")
    for k in np.unique(np.linspace(0, len(tasks) - 1, 8).astype(int)):
        print(f"[gpu] packed forms {shape} task {k}", flush=True)
        bufs, meta, _, sz = oracle.task_packed(t, so, tasks[k], False)
        dev = {n: DevBuf.from_array(bufs[n]) for n in names}
        dims = [int(t.tiles[b]) for b in tasks[k]]
        ev = [DevBuf.from_array(evl[offs[b]:offs[b] + t.tiles[b]]) for b in tasks[k]]
        nb = int(np.prod([(d + 3) // 4 for d in dims]))
        most = {n: sz[n] // (9 if n.startswith("s1") else sz["max_" + n[:2]]) for n in names}
        out = []
        for noalloc in (False, True):
            part = DevBuf(16 * nb)
            xt.fully_fused_ccsd_t_gpu(st.h, nb, dims, [dev[n].ptr for n in names], meta, t.noab, t.nvab, most,
                                      [e.ptr for e in ev], part.ptr, noalloc=noalloc)
            st.sync()
            out.append(part.to_array(2 * nb))
            part.free()
        assert np.array_equal(out[0], out[1])
        got = fac[k] * np.sum(out[0][:nb]), fac[k] * np.sum(out[0][nb:])
        assert close(got[0], ref[k, 0]) and close(got[1], ref[k, 1]), (k, dims, got, ref[k])
        for b in list(dev.values()) + ev:
            b.free()
    st.destroy()
