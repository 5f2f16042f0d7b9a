"""fq_run captured into a HIP graph on a caller's stream: deeper than the run before it,
replayed between eager runs of other depths and schedules on the same state (whose
scratch grows), each replay against the same run on a state of its own.

The same kernels on the same plans, but a captured run may make its phase tables one
by one: 1e-12 (complex128) and 1e-5 (complex64) as for any two routes.
"""
import numpy as np
import pytest
import torch

from forqaoa import Graph, State
from forqaoa import graphs as G

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-12, "c64": 1e-5}


@pytest.mark.parametrize("N,dtype,schedule,P", [
    # one launch for all layers; two passes; a table for each pass; chunks on two streams
    (12, "c128", "fused", 7), (16, "c128", "fused", 7), (16, "c64", "z2", 8), (20, "c64", "fused", 40),
    (22, "c128", "fused", 40), (25, "c64", "fused", 7), (26, "c64", "fused", 6), (14, "c128", "reference", 6),
])
def test_captured_run(N, dtype, schedule, P):
    print(f"captured run N={N} {dtype} {schedule} P={P}", flush=True)
    edges = G.gnp(N, 0.4, 9300 + N, "uniform")
    g, b = G.angles(P, 9400 + N)
    # (the reference schedule relabels its graph: a graph of its own for each run)
    gr, other = Graph(N, edges), Graph(N, edges)
    st, alone = State(N, C=10, dtype=dtype), State(N, C=10, dtype=dtype)
    alone.run(other, g, b, schedule)
    want = alone.copy_out().astype(np.complex128)
    alone.destroy()
    eager = "fused" if schedule == "reference" else schedule
    s = torch.cuda.Stream()
    st.set_stream(s.cuda_stream)
    warm = 4 if P % 2 == 0 else 5   # (plans of either parity's passes)
    st.run(gr, g[:warm], b[:warm], eager)
    st.sync()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        st.run(gr, g, b, schedule)
    deep = G.angles(P + 25, 9500 + N)
    for rep in range(4):
        st.run(gr, *deep, eager)
        if rep == 2:
            st.rotationCompressionWeighted(0.3, gr, False)
        e = st.expect_cut(gr)
        assert np.isfinite(e[0])
        with torch.cuda.stream(s):
            graph.replay()
        s.synchronize()
        got = st.copy_out().astype(np.complex128)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) < TOL[dtype], rep
    del graph
    st.destroy()
    gr.destroy()
    other.destroy()


@pytest.mark.parametrize("N,dtype,schedule,P", [
    # a layer a launch, as an eager run of one layer left room for one table; two passes
    (12, "c128", "fused", 5), (11, "c64", "z2", 4), (14, "c128", "fused", 5), (16, "c64", "z2", 4),
])
def test_captured_run_on_weights_not_seen_before(N, dtype, schedule, P):
    """Its plans are uploaded by each replay; eager runs on the same weights, before the
    first replay and between them, have their own."""
    print(f"captured run with new plans N={N} {dtype} {schedule} P={P}", flush=True)
    edges = G.gnp(N, 0.4, 9600 + N, "uniform")
    u, v, w = edges[0]
    changed = [(u, v, w + 0.75)] + list(edges[1:])
    g, b = G.angles(P, 9700 + N)
    alone, fresh = State(N, C=10, dtype=dtype), Graph(N, changed)
    alone.run(fresh, g, b, schedule)
    want = alone.copy_out().astype(np.complex128)
    alone.destroy()
    fresh.destroy()
    st, gr = State(N, C=10, dtype=dtype), Graph(N, edges)
    s = torch.cuda.Stream()
    st.set_stream(s.cuda_stream)
    st.run(gr, g[:1], b[:1], schedule)
    st.sync()
    gr.addEdgeTo2DGraph(u, v, w + 0.75)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        st.run(gr, g, b, schedule)
    for rep in range(3):
        st.run(gr, g, b, schedule)
        got = st.copy_out().astype(np.complex128)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) < TOL[dtype], rep
        st.run(gr, g[:1], b[:1], schedule)
        with torch.cuda.stream(s):
            graph.replay()
        s.synchronize()
        got = st.copy_out().astype(np.complex128)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) < TOL[dtype], rep
    del graph
    st.destroy()
    gr.destroy()
