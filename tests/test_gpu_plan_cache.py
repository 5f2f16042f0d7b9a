"""A graph whose plan cache is full of <C> plans of other weights (smaller than the
plans of a run): runs, gradients and slabs on new weights against a fresh graph.

The same kernels on the same plans: equal to the last bit.
"""
import numpy as np
import pytest

from forqaoa import Graph, State
from forqaoa import graphs as G
from forqaoa.serve import Slab

pytestmark = pytest.mark.gpu


def _slab(N, dtype, gr, g, b):
    sb = Slab(N, 2, dtype, "fused")
    req = type("R", (), {"gammas": g, "betas": b})()
    sb.assign(0, gr, req)
    for _ in g:
        sb.step()
        while sb.poll():
            pass
    sb.collect()
    sb.destroy()
    return req.expect, req.norm2


@pytest.mark.parametrize("N,dtype,small", [(22, "c128", 62), (22, "c128", 63), (23, "c64", 63), (25, "c64", 63)])
def test_full_plan_cache(N, dtype, small):
    print(f"full plan cache N={N} {dtype}", flush=True)
    edges = G.gnp(N, 0.5, 9000 + N, "uniform")
    g, b = G.angles(3, 9100 + N)
    used, st = Graph(N, edges), State(N, C=10, dtype=dtype)
    for i in range(small):
        used.add_edge(0, N - 1, 1.0 + i)
        st.expect_cut(used)
    for i in range(2):
        fresh = Graph(N, edges)
        for gr in (used, fresh):
            gr.add_edge(0, N - 1, 0.25 + i)
        st.run(used, g, b)
        got, e = st.copy_out(), st.expect_cut(used)
        grad = st.backward(used, g, b)
        s = _slab(N, dtype, used, g, b)
        st.run(fresh, g, b)
        assert np.array_equal(got, st.copy_out())
        assert e == st.expect_cut(fresh)
        want = st.backward(fresh, g, b)
        assert grad[0] == want[0] and np.array_equal(grad[1], want[1]) and np.array_equal(grad[2], want[2])
        assert s == _slab(N, dtype, fresh, g, b)
        fresh.destroy()
    st.destroy()
    used.destroy()
