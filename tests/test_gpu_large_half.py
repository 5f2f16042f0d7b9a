"""Half states of 64 GiB, where every pass takes its tiles by XCD (MixArgs::by_xcd): the
amplitudes and <C> of the fused schedule, which runs other passes over the same qubits.

Tolerance: both within (N + 2) P roundings of a unit-norm state, so the vector of the
sampled amplitudes and <C> agree to 1e-12 and 1e-5 with a margin.
"""
import numpy as np
import pytest

from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dtype,P", [(33, "c64", 3), (33, "c64", 2), (32, "c128", 3)])
def test_half_state_vs_fused(N, dtype, P):
    print(f"half state N={N} {dtype} P={P}", flush=True)
    g = Graph(N, G.gnp(N, 0.3, 8600 + N, "uniform"))
    gm, bt = G.angles(P, 8700 + N)
    idx = np.random.default_rng(N).integers(0, 1 << N, size=8192, dtype=np.uint64)
    st = State(N, C=13, dtype=dtype)
    got = []
    for schedule in ("z2", "fused"):
        st.run(g, gm, bt, schedule)
        got.append((st.gather(idx, logical=True), st.expect_cut(g)))
    st.destroy()
    g.destroy()
    (a, ea), (b, eb) = got
    tol = {"c128": 1e-12, "c64": 1e-5}[dtype]
    assert np.linalg.norm(a - b) / np.linalg.norm(b) < tol
    assert ea[0] == pytest.approx(eb[0], rel=tol)
    assert ea[1] == pytest.approx(1.0, abs=tol)
