"""Small states in one launch (k_solo) and the narrow plans next to them: both ends
of the sizes, odd and even depths (which layout the state is stored from), more
layers than one launch takes (64), weights with and without an edge inside the
registers, every schedule, against the oracle.

Tolerance: (N + 1) roundings per layer and amplitude at most, in quadrature over
the amplitudes of a unit-norm state: eps sqrt(13 * 130) = 41 eps, under 1e-13 and
5e-6; 1e-12 and 1e-5 with the oracle's own rounding.
"""
import numpy as np
import pytest

import pyoracle as O
from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dtype,P", [
    (8, "c128", 2), (9, "c128", 1), (9, "c128", 2), (10, "c128", 3), (11, "c128", 4), (12, "c128", 1), (12, "c128", 5),
    (13, "c128", 1), (13, "c128", 2), (10, "c128", 64), (9, "c128", 65), (11, "c128", 130),
    (9, "c64", 2), (10, "c64", 1), (10, "c64", 2), (11, "c64", 3), (12, "c64", 4), (13, "c64", 1), (13, "c64", 2),
    (14, "c64", 1), (14, "c64", 3), (12, "c64", 64), (10, "c64", 66),
])
def test_small_states(N, dtype, P):
    for schedule, density, weights in (("fused", 0.5, "uniform"), ("z2", 0.1, "int16"), ("reference", 0.9, "uniform")):
        print(f"small state N={N} {dtype} P={P} {schedule}", flush=True)
        edges = G.gnp(N, density, 8000 + N + P, weights)
        gm, bt = G.angles(P, 8100 + N + P)
        C = max(1, N // 2)
        sv, qmap, W = O.run_weighted(N, C, edges, gm, bt)
        st, g = State(N, C=C, dtype=dtype), Graph(N, edges)
        for _ in range(2 if schedule != "reference" else 1):
            st.run(g, gm, bt, schedule)
        got = st.copy_out(logical=True).astype(np.complex128)
        ex, _ = st.expect_cut(g)
        st.destroy()
        g.destroy()
        want = O.to_logical(sv, qmap)
        tol = {"c128": 1e-12, "c64": 1e-5}[dtype]
        err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
        assert err < tol, (schedule, err)
        e = O.expect_cut(sv, W)
        assert abs(ex - e) <= tol * max(1.0, abs(e))
