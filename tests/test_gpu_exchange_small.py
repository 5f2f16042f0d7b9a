"""Exchanges of small states, a thread per amplitude, up to the size from which they go in
tiles: bitwise against the axis permutation in numpy, and the exchanges of scattered
pairs that end the reference schedule against its single steps (amplitudes within
(N + 2) P roundings of the unit-norm state: 1e-12 and 1e-5 with a margin).
"""
import numpy as np
import pytest

import refmath as R
from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("N", [2, 3, 8, 9, 16, 17, 18, 19])
def test_exchange_bitwise(N, dtype):
    print(f"small exchange N={N} {dtype}", flush=True)
    rng = np.random.default_rng(N)
    v = (rng.normal(size=1 << N) + 1j * rng.normal(size=1 << N)).astype(np.complex128 if dtype == "c128" else np.complex64)
    st = State(N, C=min(N, 8), dtype=dtype)
    for out, inn, k in ((0, N // 2, N // 2), (0, N - 1, 1), (N - 2, N - 1, 1), (N // 4, N // 2, max(1, N // 4)), (0, 1, 1)):
        st.copy_in(v)
        st.swap_conti(out, inn, k)
        v = R.axis_swap_blocks(v, N, out, inn, k)
        np.testing.assert_array_equal(st.copy_out(), v)
    st.destroy()


@pytest.mark.parametrize("N,C,dtype", [(11, 3, "c128"), (16, 5, "c128"), (17, 5, "c128"), (17, 4, "c64"), (18, 4, "c64"), (13, 1, "c64")])
def test_reference_schedule_vs_single_steps(N, C, dtype):
    print(f"reference schedule N={N} C={C} {dtype}", flush=True)
    edges, (gm, bt) = G.gnp(N, 0.5, 5200 + N, "uniform"), G.angles(3, 5300 + N)
    out = []
    for timing in (True, False):
        st, g = State(N, C=C, dtype=dtype), Graph(N, edges)
        st.timing(timing)
        st.run(g, gm, bt, "reference")
        out.append((st.copy_out().astype(np.complex128), list(st.qubit_map()), np.array(g.weights())))
        st.destroy()
        g.destroy()
    assert out[0][1] == out[1][1]
    np.testing.assert_array_equal(out[0][2], out[1][2])
    assert np.linalg.norm(out[0][0] - out[1][0]) < {"c128": 1e-12, "c64": 1e-5}[dtype]
