"""The pair passes of the gradient on compile-time phases (fq_pair.hip) at the
edges of their plans: the first and last size of each tile width, two and three
passes, odd and even depths (which pass the walk starts on), chunked walks, and
more passes than one phase-table launch takes.

Against the general pair passes (FQ_LAYER_PIPE=0: other tiles, other order) on
the same angles, and against central differences of the oracle's <C> at the
smallest sizes.  Tolerances on max |difference| / max(1, |g|): the sums are
FP64 over amplitudes with under 100 roundings each, times the size of Cut and S
(under 1e3 here): 1e-16 * 1e2 * 1e3 = 1e-11, 1e-10 with a margin; complex64
(1e-7, in quadrature over amplitudes) 1e-4, as for the general passes.
"""
import os

import numpy as np
import pytest

import pyoracle as O
from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-10, "c64": 1e-4}


def _grad(N, dtype, edges, g, b, schedule, general):
    old = os.environ.pop("FQ_LAYER_PIPE", None)
    if general:
        os.environ["FQ_LAYER_PIPE"] = "0"
    try:
        st, gr = State(N, C=min(N, 10), dtype=dtype), Graph(N, edges)
        st.run(gr, g, b, schedule)
        out = st.backward(gr, g, b)
        st.destroy()
        gr.destroy()
    finally:
        os.environ.pop("FQ_LAYER_PIPE", None)
        if old is not None:
            os.environ["FQ_LAYER_PIPE"] = old
    return out


@pytest.mark.parametrize("N,dtype,P", [
    # complex128: 9-qubit tiles from N=10, then 10, 11, 12 wide, three passes, chunks
    (10, "c128", 1), (11, "c128", 2), (15, "c128", 3), (16, "c128", 2), (17, "c128", 1), (18, "c128", 2),
    (19, "c128", 3), (20, "c128", 2), (21, "c128", 3), (22, "c128", 2), (22, "c128", 3), (24, "c128", 2),
    (25, "c128", 3), (26, "c128", 2),
    # complex64: 10-qubit tiles from N=11, then 11, 12, 13 wide, three passes, chunks
    (11, "c64", 1), (12, "c64", 2), (16, "c64", 3), (17, "c64", 2), (18, "c64", 1), (19, "c64", 2),
    (20, "c64", 3), (21, "c64", 2), (22, "c64", 3), (23, "c64", 2), (23, "c64", 3), (24, "c64", 2),
    (26, "c64", 3), (27, "c64", 2),
    # more cost passes than one phase-table launch takes
    (14, "c128", 67), (16, "c64", 66),
])
def test_pair_passes_vs_general(N, dtype, P):
    print(f"gradient N={N} {dtype} P={P}", flush=True)
    edges = G.gnp(N, 0.4, 4600 + N + P, "uniform")
    g, b = G.angles(P, 4700 + N + P)
    schedule = "z2" if (N + P) % 3 == 0 else "fused"
    e, gg, gb = _grad(N, dtype, edges, g, b, schedule, False)
    e0, gg0, gb0 = _grad(N, dtype, edges, g, b, schedule, True)
    d0 = np.concatenate([gg0, gb0])
    err = float(np.max(np.abs(np.concatenate([gg, gb]) - d0))) / max(1.0, float(np.max(np.abs(d0))))
    print(f"  max difference / max(1, |g|) {err:.2e}", flush=True)
    assert abs(e - e0) / abs(e0) < {"c128": 1e-12, "c64": 1e-5}[dtype]
    assert err < TOL[dtype]


@pytest.mark.parametrize("N,dtype,P", [(10, "c128", 3), (11, "c64", 2), (12, "c128", 2)])
def test_pair_passes_vs_oracle(N, dtype, P):
    print(f"gradient N={N} {dtype} P={P} against the oracle", flush=True)
    edges = G.gnp(N, 0.5, 4800 + N, "uniform")
    # angles whose RX takes every branch of the butterfly form (small, near pi, negative, beyond 2 pi)
    g = np.array([0.3, -1.2, 0.7])[:P]
    b = np.array([3.1, -0.4, 7.0])[:P]
    _, gg, gb = _grad(N, dtype, edges, g, b, "fused", False)

    def f(x, y):
        sv, _, W = O.run_weighted(N, 4, edges, x, y)
        return O.expect_cut(sv, W)

    h, want = 1e-4, []
    for k in range(2 * P):
        d = h * np.eye(2 * P)[k]
        want.append((f(g + d[:P], b + d[P:]) - f(g - d[:P], b - d[P:])) / (2 * h))
    err = float(np.max(np.abs(np.concatenate([gg, gb]) - want))) / max(1.0, float(np.max(np.abs(want))))
    print(f"  max difference / max(1, |g|) {err:.2e}", flush=True)
    # (the central difference itself is accurate to ~1e-9)
    assert err < {"c128": 1e-7, "c64": 1e-4}[dtype]
