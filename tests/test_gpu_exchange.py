"""Qubit exchanges (k_exchange) and the reference schedule without its single steps.

* fq_swap_conti at the edges of the tile widths (2^8 or fewer amplitudes,
  2^10, 2^12), blocks low, high and adjacent, one qubit to half of them:
  bitwise against the axis permutation in numpy.
* FQ_SCHED_REFERENCE: with timing on it runs step by step, otherwise as fused
  layers and the product of its transpositions.  Chunk widths from 1 (a
  permutation of single qubits) to N (no transposition), so that the product is
  the identity, one exchange or two, of runs and of scattered pairs, from a
  state in the identity layout and from one that is already permuted.  Layout
  and graph exactly; amplitudes within (N + 2) P roundings of the unit-norm
  state: 1e-12 and 1e-5 with a margin.
"""
import numpy as np
import pytest

import refmath as R
from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu


def _random(N, dtype, seed):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=1 << N) + 1j * rng.normal(size=1 << N)
    return (v / np.linalg.norm(v)).astype(np.complex128 if dtype == "c128" else np.complex64)


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("N,out,inn,k", [
    (2, 0, 1, 1), (5, 1, 3, 2), (7, 0, 4, 3), (8, 0, 4, 4), (9, 2, 6, 3), (10, 0, 9, 1), (10, 5, 7, 2),
    (11, 0, 5, 5), (12, 6, 9, 3), (13, 0, 7, 6), (21, 0, 12, 9), (22, 9, 16, 6), (23, 1, 22, 1),
    (24, 0, 12, 12), (24, 11, 13, 2), (25, 0, 13, 12), (25, 5, 20, 1), (24, 3, 14, 7),
])
def test_exchange_bitwise(N, out, inn, k, dtype):
    print(f"exchange N={N} {dtype} [{out},+{k}) [{inn},+{k})", flush=True)
    st = State(N, C=min(N, 8), dtype=dtype)
    v = _random(N, dtype, N + k)
    st.copy_in(v)
    st.swap_conti(out, inn, k)
    got = st.copy_out()
    st.destroy()
    np.testing.assert_array_equal(got, R.axis_swap_blocks(v, N, out, inn, k))


@pytest.mark.parametrize("N,C,P,dtype", [
    (1, 1, 2, "c128"), (3, 1, 2, "c128"), (5, 2, 3, "c64"), (9, 1, 4, "c128"), (9, 4, 1, "c64"), (12, 5, 2, "c128"),
    (12, 6, 2, "c64"), (13, 13, 2, "c128"), (14, 3, 5, "c128"), (16, 8, 2, "c128"), (17, 1, 3, "c64"),
    (17, 7, 3, "c128"), (18, 5, 4, "c64"), (20, 12, 5, "c128"), (21, 9, 6, "c64"), (24, 13, 2, "c128"),
    (25, 14, 3, "c64"), (25, 6, 2, "c64"),
])
def test_reference_schedule_vs_single_steps(N, C, P, dtype):
    print(f"reference schedule N={N} C={C} P={P} {dtype}", flush=True)
    edges = G.gnp(N, 0.5, 5000 + N + C, "uniform") if N > 1 else []
    gm, bt = G.angles(P, 5100 + N + P)
    out = []
    for timing in (True, False):
        st, g = State(N, C=C, dtype=dtype), Graph(N, edges)
        for _ in range(2):   # the second run starts from the permuted layout
            st.timing(timing)
            st.run(g, gm, bt, "reference")
            out.append((st.copy_out().astype(np.complex128), list(st.qubit_map()), np.array(g.weights())))
        st.destroy()
        g.destroy()
    for a, b in zip(out[:2], out[2:]):
        assert a[1] == b[1]
        np.testing.assert_array_equal(a[2], b[2])
        err = float(np.linalg.norm(a[0] - b[0]))
        assert err < {"c128": 1e-12, "c64": 1e-5}[dtype], err
