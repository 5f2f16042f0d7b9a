"""The general kernels, where the default plans no longer come: boundary passes of
tiles narrower than fq_mix.h has (k_tile), its tile orders, and the pipelined walk
back of the general pair pass, which the gradients of the largest states take (from
N=31 complex128, 32 complex64).

States against the oracle within 1e-12 / 1e-5, as for the other plans.  A tile order
changes which work-group takes a tile, not what is done with it: equal to the last
bit.  Gradients against fq_pair.hip's with that file's tolerances: on max
|difference| / max(1, |g|) 1e-10 (FP64 sums, under 100 roundings each, times Cut and S
below 1e3: 1e-11 with a margin) and 1e-4.
"""
import os

import numpy as np
import pytest

import pyoracle as O
from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-12, "c64": 1e-5}
GRAD_TOL = {"c128": 1e-10, "c64": 1e-4}
KNOBS = ["FQ_TILE_Q", "FQ_TILE_ORDER", "FQ_PASS_BLOCK", "FQ_CARRIER_GATES", "FQ_LAYER_PIPE"]


@pytest.fixture
def knobs(monkeypatch):
    def set_to(**env):
        for k in KNOBS:
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)

    set_to()
    return set_to


def _state(N, dtype, edges, g, b, schedule):
    st, gr = State(N, C=min(N, 10), dtype=dtype), Graph(N, edges)
    try:
        st.run(gr, g, b, schedule)
        return st.copy_out(logical=True).astype(np.complex128), st.expect_cut(gr)[0]
    finally:
        st.destroy()
        gr.destroy()


@pytest.mark.parametrize("schedule", ["fused", "z2"])
@pytest.mark.parametrize("N,dtype,Q,P", [
    # two passes a layer (the half state in layer order), three and four; the narrowest
    # tiles, whose work-groups are half a wave and less
    (13, "c128", 8, 3), (16, "c128", 8, 2), (20, "c128", 8, 3), (12, "c128", 6, 3),
    (14, "c64", 9, 3), (17, "c64", 9, 4), (20, "c64", 9, 3), (13, "c64", 7, 2),
])
def test_boundary_passes_of_narrow_tiles(knobs, N, dtype, Q, P, schedule):
    print(f"general boundary passes N={N} {dtype} Q={Q} {schedule}", flush=True)
    edges = G.gnp(N, 0.5, 7300 + N + Q, "uniform")
    g, b = G.angles(P, 7400 + N + Q)
    b[0] = 2.9   # RX beyond the butterfly's first branch
    sv, qmap, W = O.run_weighted(N, min(N, 6), edges, g, b)
    want, e = O.to_logical(sv, qmap), O.expect_cut(sv, W)
    knobs(FQ_TILE_Q=str(Q))
    got, ex = _state(N, dtype, edges, g, b, schedule)
    assert np.linalg.norm(got - want) < TOL[dtype] * np.linalg.norm(want)
    assert abs(ex - e) < TOL[dtype] * abs(e)


@pytest.mark.parametrize("N,dtype,Q", [(23, "c128", 8), (24, "c64", 9)])
@pytest.mark.parametrize("order", ["0", "1", "3"])
def test_tile_orders_are_equal(knobs, N, dtype, Q, order):
    # more tiles than work-groups fit, so that the orders differ: the cost phase alone
    # (12-qubit tiles), then passes with and without it
    print(f"tile order {order} N={N} {dtype}", flush=True)
    edges = G.gnp(N + 1, 0.4, 7500, "uniform")
    g, b = G.angles(2, 7501)
    out = []
    for o in ("2", order):
        knobs(FQ_TILE_ORDER=o)
        st, gr = State(N + 1, C=10, dtype=dtype), Graph(N + 1, edges)
        st.rotationCompressionWeighted(float(g[0]), gr, True)
        st.rotationCompressionWeighted(float(g[1]), gr, False)
        v = st.gather(np.arange(0, 1 << (N + 1), 977))
        st.destroy()
        gr.destroy()
        knobs(FQ_TILE_ORDER=o, FQ_TILE_Q=str(Q))
        small = [(u, w, x) for u, w, x in edges if w < N]
        out.append((v, *_state(N, dtype, small, g, b, "fused"), *_state(N, dtype, small, g, b, "z2")))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("N,dtype,P", [(22, "c128", 3), (24, "c128", 2), (21, "c64", 3), (23, "c64", 2), (24, "c64", 1)])
def test_pipelined_general_walk_back(knobs, N, dtype, P):
    print(f"general walk back N={N} {dtype} P={P}", flush=True)
    edges = G.gnp(N, 0.4, 7600 + N + P, "uniform")
    g, b = G.angles(P, 7700 + N + P)

    def grad():
        st, gr = State(N, C=10, dtype=dtype), Graph(N, edges)
        st.run(gr, g, b, "fused")
        out = st.backward(gr, g, b)
        st.destroy()
        gr.destroy()
        return out

    e0, gg0, gb0 = grad()
    knobs(FQ_PASS_BLOCK="2")   # the default's value, but no plan of fq_pair.hip
    e1, gg1, gb1 = grad()
    tol = GRAD_TOL[dtype]
    assert abs(e1 - e0) < tol * max(1.0, abs(e0))
    for x, y in ((gg0, gg1), (gb0, gb1)):
        assert np.max(np.abs(x - y)) < tol * max(1.0, np.max(np.abs(x)))
