"""A graph that changes while slab slots run it: each slot's next layer takes the new
weights, wherever the slot is, and a copy-out in between shows the layers run so far
with theirs.

Against the layers gate by gate, each with the weights it ran with.  Tolerance as for
packed slabs: both are off by (N + 2) P roundings of a unit-norm state at most (and
three passes more): 1e-12 and 1e-5 with a margin.
"""
import numpy as np
import pytest

from forqaoa import Graph, State
from forqaoa import graphs as G
from forqaoa.serve import Slab

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-12, "c64": 1e-5}


def _layers(N, dtype, weights, g, b):
    """Layer p with the graph of edge list weights[p]; the state and the last graph's <C>."""
    st = State(N, C=min(N, 10), dtype=dtype)
    for p, edges in enumerate(weights):
        gr = Graph(N, edges)
        st.rotationCompressionWeighted(float(g[p]), gr, p == 0)
        st.multiRotateX(list(range(N)), N, float(b[p]))
        e = st.expect_cut(gr)
        gr.destroy()
    v = st.copy_out().astype(np.complex128)
    st.destroy()
    return v, e


@pytest.mark.parametrize("N,dtype,schedule", [
    # the general kernel; packed slots, both types and schedules; slots one by one
    (8, "c128", "fused"), (10, "c128", "fused"), (14, "c128", "fused"), (16, "c64", "z2"), (18, "c128", "z2"),
    (20, "c64", "fused"), (22, "c128", "z2"), (23, "c64", "z2"), (24, "c64", "z2"), (25, "c64", "fused"),
    (25, "c128", "z2"),
])
def test_changed_graph_counts_from_the_next_layer(N, dtype, schedule):
    print(f"changed graph N={N} {dtype} {schedule}", flush=True)
    base = G.gnp(N, 0.4, 8000 + N, "uniform")
    versions = [list(base)]
    for i in range(3):   # a changed weight, a new edge or one that goes
        e = list(versions[-1])
        u, v, w = e[i]
        e[i] = (u, v, w + 0.5 if i != 1 else 0.0)
        versions.append(e)
    P = [4, 3]
    ang = [G.angles(p, 8100 + N + p) for p in P]
    ang[0][1][1] = 2.9   # RX beyond the butterfly's first branch
    gr, sb = Graph(N, base), Slab(N, 2, dtype, schedule)
    ran = [[], []]   # version each slot's layers ran with
    reqs = [type("R", (), {"gammas": g, "betas": b})() for g, b in ang]
    now = 0
    for step in range(5):
        if step == 0:
            sb.assign(0, gr, reqs[0])
        if step == 1:    # enters as the other one goes on
            sb.assign(1, gr, reqs[1])
        if step in (1, 2, 3):
            u, v, w = versions[now + 1][now]
            gr.add_edge(u, v, w)
            now += 1
            if step == 2:    # changed, and no step since
                got = sb.copy_out(0, dtype).astype(np.complex128)
                want, _ = _layers(N, dtype, [versions[i] for i in ran[0]], *ang[0])
                assert np.linalg.norm(got - want) / np.linalg.norm(want) < TOL[dtype]
        running = [k for k in sb.slot_req if len(ran[k]) < P[k]]
        sb.step()
        for k in running:
            ran[k].append(now)
        while sb.poll():
            pass
        done = [k for k in running if len(ran[k]) == P[k]]
        got = {k: sb.copy_out(k, dtype).astype(np.complex128) for k in done}
        sb.collect()
        for k in done:
            want, (e, n2) = _layers(N, dtype, [versions[i] for i in ran[k]], *ang[k])
            assert np.linalg.norm(got[k] - want) / np.linalg.norm(want) < TOL[dtype], k
            assert reqs[k].expect == pytest.approx(e, rel=TOL[dtype])
            assert reqs[k].norm2 == pytest.approx(n2, abs=TOL[dtype])
    assert [len(r) for r in ran] == P
    sb.destroy()
    gr.destroy()
