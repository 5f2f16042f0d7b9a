"""The compile-time tile passes (fq_mix.hip) at the edges of their cases.

* RX on every kind of target set of a full-width tile: register bits only, 1
  to 3 exchanges, one more bit by lane operations, single bits, sets that skip
  bits, contiguous and strided tiles, one tile and several -- against RX
  applied in numpy to the same random state.
* Chunked runs (states beyond the memory-side cache): the smallest such sizes,
  full and half state, odd and even depths (the half state's first pass is the
  mirror pass for even ones), against the same run without chunks and, once
  per type, against the oracle.

Tolerances: every RX is one FMA per component, so a state of unit norm is off
by at most about (gates) x eps in the 2-norm, and the phases add a few eps per
layer: under 200 eps here, 1e-13 / 3e-5 with a margin of 2 to 4.
"""
import os

import numpy as np
import pytest

import pyoracle as O
from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-13, "c64": 3e-5}


def _rx(v, q, beta):
    a = v.reshape(-1, 2, 1 << q)
    x, y = a[:, 0].copy(), a[:, 1].copy()
    c, s = np.cos(beta / 2), -1j * np.sin(beta / 2)
    a[:, 0] = c * x + s * y
    a[:, 1] = s * x + c * y


SETS = [[12], [0], [4], [3], [9, 10, 11, 12], [8], list(range(5, 13)), list(range(4, 13)), list(range(1, 13)),
        list(range(0, 13)), [0, 5, 12], [2, 4, 9], [4, 8], [0, 1], [1, 2, 3, 4],
        [13], [14, 15], [12, 13], [0, 15], list(range(6, 16)), [3, 7, 13, 15]]


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("N", [14, 16])
def test_rx_sets(N, dtype):
    Q = 13 if dtype == "c128" else 14
    sets = SETS + ([list(range(3, 14)), list(range(4, 14)), list(range(0, 14))] if dtype == "c64" else [])
    rng = np.random.default_rng(N)
    st = State(N, C=Q, dtype=dtype)
    for k, targets in enumerate(sets):
        if max(targets) >= N:
            continue
        v = rng.normal(size=1 << N) + 1j * rng.normal(size=1 << N)
        v /= np.linalg.norm(v)
        beta = float(rng.uniform(-3, 3))
        print(f"N={N} {dtype} RX({beta:.3f}) on {targets}", flush=True)
        st.copy_in(v.astype(st.np_dtype))
        st.multi_rx(targets, beta)
        got = st.copy_out().astype(np.complex128)
        for q in targets:
            _rx(v, q, beta)
        assert np.linalg.norm(got - v) < TOL[dtype], targets
    st.destroy()


@pytest.fixture
def chunk_env():
    old = os.environ.get("FQ_CHUNK")
    yield
    os.environ.pop("FQ_CHUNK", None)
    if old is not None:
        os.environ["FQ_CHUNK"] = old


def _state(N, dtype, schedule, P, edges, chunk):
    os.environ.pop("FQ_CHUNK", None)
    if chunk is not None:
        os.environ["FQ_CHUNK"] = chunk
    gm, bt = G.angles(P, 4100 + N + P)
    st, g = State(N, C=10, dtype=dtype), Graph(N, edges)
    st.run(g, gm, bt, schedule)
    v = st.copy_out(logical=True)
    st.destroy()
    g.destroy()
    return v, gm, bt


@pytest.mark.parametrize("N,dtype,schedule,P,oracle", [
    (25, "c128", "fused", 1, False), (25, "c128", "fused", 2, False), (25, "c128", "fused", 3, True),
    (26, "c64", "fused", 3, True), (26, "c128", "z2", 1, False), (26, "c128", "z2", 2, True),
    (26, "c128", "z2", 3, False), (27, "c64", "z2", 2, False), (27, "c64", "z2", 3, False),
])
def test_chunked_runs(chunk_env, N, dtype, schedule, P, oracle):
    print(f"chunked N={N} {dtype} {schedule} P={P}", flush=True)
    edges = G.gnp(N, 0.4, 4200 + N, "uniform")
    got, gm, bt = _state(N, dtype, schedule, P, edges, None)
    ref, _, _ = _state(N, dtype, schedule, P, edges, "0")
    norm = np.linalg.norm(ref)
    # the two orders apply the same gates with different tilings: both errors add
    assert np.linalg.norm(got - ref) / norm < {"c128": 1e-12, "c64": 3e-5}[dtype]
    if oracle:
        del ref
        sv, qmap, _ = O.run_weighted(N, 10, edges, gm, bt)
        want = O.to_logical(sv, qmap)
        err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
        print(f"  relative L2 error vs oracle {err:.2e}", flush=True)
        assert err < {"c128": 1e-12, "c64": 1e-5}[dtype]


@pytest.mark.parametrize("N,dtype,schedule,P", [
    # the ends of each tile width of the two-pass plans (complex128 9..13,
    # complex64 10..14 qubits), and two passes over 64 B runs
    (14, "c128", "fused", 2), (15, "c128", "z2", 1), (15, "c128", "z2", 2), (16, "c128", "fused", 3),
    (17, "c128", "fused", 2), (18, "c128", "z2", 3), (19, "c128", "fused", 2), (21, "c128", "fused", 3),
    (22, "c128", "z2", 2), (23, "c128", "z2", 3), (24, "c128", "fused", 2),
    (15, "c64", "fused", 2), (16, "c64", "z2", 2), (17, "c64", "fused", 3), (18, "c64", "z2", 1),
    (20, "c64", "fused", 2), (21, "c64", "fused", 3), (22, "c64", "z2", 2), (23, "c64", "z2", 3),
    (23, "c64", "fused", 2), (25, "c64", "fused", 3),
    # more cost passes than one phase-table launch takes
    (14, "c128", "fused", 66), (16, "c64", "z2", 65),
])
def test_two_pass_plans(N, dtype, schedule, P):
    print(f"two passes N={N} {dtype} {schedule} P={P}", flush=True)
    edges = G.gnp(N, 0.5, 4400 + N + P, ["uniform", "int16"][P % 2])
    gm, bt = G.angles(P, 4500 + N + P)
    sv, qmap, W = O.run_weighted(N, min(N, 8), edges, gm, bt)
    want = O.to_logical(sv, qmap)
    st, g = State(N, C=min(N, 8), dtype=dtype), Graph(N, edges)
    st.run(g, gm, bt, schedule)
    got = st.copy_out(logical=True).astype(np.complex128)
    ex, _ = st.expect_cut(g)
    st.destroy()
    g.destroy()
    err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    rel = abs(ex - O.expect_cut(sv, W)) / abs(O.expect_cut(sv, W))
    print(f"  relative L2 error vs oracle {err:.2e}, <C> {rel:.2e}", flush=True)
    # (N + 2) roundings per layer and amplitude at most, in quadrature
    tol = {"c128": 1e-12, "c64": 1e-5}[dtype]
    assert err < tol and rel < tol
