"""<C> by the last work-group, and the streams and result pages that states share.

* fq_expect_cut adds up its partials in the last work-group up to 1,024 of them
  (N = 22) and in a second launch beyond; fq_expect_cut_static always takes two
  launches.  Same order of additions: equal to the last bit, call after call.
* more states alive at once than idle streams are kept, in several threads,
  made and destroyed twice, so that streams and pages change hands: every <C>
  and gradient equal to the last bit to that of one state alone.
"""
import threading

import numpy as np
import pytest

from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("N", [1, 3, 8, 11, 12, 13, 21, 22, 23])
def test_expect_equals_two_launches(N, dtype):
    print(f"<C> N={N} {dtype}", flush=True)
    edges = G.gnp(N, 0.5, 7000 + N, "uniform") if N > 1 else []
    gm, bt = G.angles(2, 7100 + N)
    st, g = State(N, C=min(N, 10), dtype=dtype), Graph(N, edges)
    st.run(g, gm, bt, "fused")
    want = st.expect_cut_static(g)
    for _ in range(3):
        assert st.expect_cut(g) == want
    st.destroy()
    g.destroy()


def test_states_in_threads_share_streams():
    N, P = 11, 3
    edges = G.gnp(N, 0.5, 7200, "uniform")
    angles = [G.angles(P, 7300 + i) for i in range(24)]

    def one(i, g):
        st = State(N, C=6, dtype="c128")
        st.run(g, *angles[i], "fused")
        return st, st.expect_cut(g), st.backward(g, *angles[i])

    def flat(r):
        return np.concatenate([r[1], [r[2][0]], r[2][1], r[2][2]])

    g = Graph(N, edges)
    want = []
    for i in range(24):
        r = one(i, g)
        want.append(flat(r))
        r[0].destroy()
    got, failed = {}, []

    def work(k):
        try:
            own = Graph(N, edges)
            for _ in range(2):
                live = [(i, one(i, own)) for i in range(k, 24, 4)]
                for i, r in live:
                    got.setdefault(i, []).append(flat(r))
                    r[0].destroy()
            own.destroy()
        except Exception as e:   # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for i in range(24):
        assert len(got[i]) == 2
        for v in got[i]:
            np.testing.assert_array_equal(v, want[i])
    g.destroy()
