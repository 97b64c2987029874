"""Both expansion kernels: pairs staged in LDS (O up to 84, output 16-byte
aligned) and element by element (the rest), against the closed-shell rule
(cd_ccsd_cs_ann.cpp:932-976) and against each other, bit for bit."""
import numpy as np
import pytest


pytestmark = pytest.mark.gpu


def _expected(s, O, V):
    t, x = s["t2"], s["t2"] - s["t2"].transpose(0, 1, 3, 2)
    so = np.zeros((2 * V, 2 * V, 2 * O, 2 * O))
    a, b = slice(0, V), slice(V, 2 * V)
    i, j = slice(0, O), slice(O, 2 * O)
    so[a, a, i, i] = so[b, b, j, j] = x
    so[a, b, i, j] = so[b, a, j, i] = t
    so[a, b, j, i] = so[b, a, i, j] = -t.transpose(0, 1, 3, 2)
    return so


@pytest.mark.parametrize("O,V", [(1, 2), (2, 3), (3, 5), (7, 6), (16, 5), (83, 3), (84, 2), (85, 2)])
@pytest.mark.parametrize("shift", [0, 8])
def test_expansion_over_both_kernels(xt, O, V, shift):
    from exachem_amd.hipmem import DevBuf, Stream
    print(f"[gpu] expand O={O} V={V} shift {shift}", flush=True)
    s = xt.synth_closed_shell(O, V, 41, 0.05, 1e-3)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling(O, V, [O], [V]), True)
    ctx.upload(s)
    want, n = _expected(s, O, V), 16 * O * O * V * V
    buf, st = DevBuf.from_array(np.full(n + 2, 7.0)), Stream()
    ctx.expand_amplitudes(None, buf.ptr.value + shift, st.h)
    st.sync()
    got = buf.to_array(n + 2)
    k = shift // 8
    assert np.array_equal(got[k:k + n], want.ravel())
    assert np.all(got[:k] == 7.0) and np.all(got[k + n:] == 7.0)  # nothing outside
    buf.free()
    st.destroy()
    ctx.close()
