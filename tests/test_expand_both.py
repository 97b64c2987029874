"""T1 and T2 written by one call, over both forms of the expansion: the same bits
as T1 and T2 alone, nothing outside either output."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("O,V", [(1, 1), (1, 2), (7, 22), (16, 33), (20, 9), (84, 2), (85, 2)])
@pytest.mark.parametrize("shift", [0, 8])
def test_one_call_for_both(xt, O, V, shift):
    from exachem_amd.hipmem import DevBuf, Stream
    print(f"[gpu] expand both O={O} V={V} shift {shift}", flush=True)
    s = xt.synth_closed_shell(O, V, 41, 0.05, 1e-3)
    ctx = xt.CCSDTriples(0)
    ctx.set_tiling(xt.Tiling(O, V, [O], [V]), True)
    ctx.upload(s)
    n1, n2, st = 4 * O * V, 16 * O * O * V * V, Stream()
    one, two = [[DevBuf.from_array(np.full(n + 2, 7.0)) for n in (n1, n2)] for _ in range(2)]
    ctx.expand_amplitudes(one[0].ptr.value + 8, one[1].ptr.value + shift, st.h)
    ctx.expand_amplitudes(two[0].ptr.value + 8, None, st.h)
    ctx.expand_amplitudes(None, two[1].ptr.value + shift, st.h)
    st.sync()
    for x, y, n in zip(one, two, (n1, n2)):
        assert np.array_equal(x.to_array(n + 2), y.to_array(n + 2))
    t1 = np.zeros((2 * V, 2 * O))
    t1[:V, :O] = t1[V:, O:] = s["t1"]
    got = one[0].to_array(n1 + 2)
    assert np.array_equal(got[1:-1], t1.ravel()) and got[0] == got[-1] == 7.0
    for b in one + two:
        b.free()
    st.destroy()
    ctx.close()
