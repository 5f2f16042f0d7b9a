"""Packed slabs on the compile-time passes (fq_slab_step): slots that enter at
different steps, so that launches mix slots of different depth and a slot's first
layer opens on either of the two passes, at the ends of each tile width; and
the first sizes whose slots run one by one.

Each request's <C>, norm and amplitudes against the same request run alone
(fq_run: other tile order, the last pass differs).  Tolerance: both are off by
(N + 2) P roundings of a unit-norm state at most: 1e-12 and 1e-5 with a margin.
"""
import numpy as np
import pytest

from forqaoa import Graph, State
from forqaoa import graphs as G
from forqaoa.serve import Slab

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-12, "c64": 1e-5}


def _alone(N, gr, g, b, dtype):
    st = State(N, C=min(N, 10), dtype=dtype)
    st.run(gr, g, b, "fused")
    e, n2 = st.expect_cut(gr)
    v = st.copy_out().astype(np.complex128)
    st.destroy()
    return e, n2, v


@pytest.mark.parametrize("N,dtype,schedule,K", [
    (10, "c128", "fused", 4), (11, "c128", "z2", 4), (14, "c128", "z2", 8), (16, "c128", "fused", 4),
    (18, "c128", "z2", 4), (20, "c128", "fused", 2), (21, "c128", "z2", 2), (22, "c128", "fused", 2),
    (23, "c128", "z2", 2),
    (11, "c64", "fused", 4), (12, "c64", "z2", 8), (16, "c64", "z2", 16), (17, "c64", "fused", 4),
    (18, "c64", "z2", 4), (20, "c64", "z2", 4), (21, "c64", "fused", 2), (22, "c64", "z2", 2),
    (23, "c64", "fused", 2), (24, "c64", "z2", 2),
])
def test_slots_that_join_at_any_step(N, dtype, schedule, K):
    print(f"packed slab N={N} {dtype} {schedule} K={K}", flush=True)
    sb = Slab(N, K, dtype, schedule)
    graphs, running, left = [], {}, []
    for i in range(K + 2):   # depths 1..4, weights with and without an edge inside the registers
        edges = G.gnp(N, [0.15, 0.6][i % 2], 6000 + 10 * N + i, ["uniform", "int16"][i % 2])
        gm, bt = G.angles(1 + i % 4, 6100 + N + i)
        graphs.append(Graph(N, edges))
        left.append((graphs[-1], gm, bt))
    for step in range(4 * (K + 2)):
        free = [k for k in range(K) if k not in running]
        # one request a step, two on every third
        for k in free[:1 + (step % 3 == 2)]:
            if left:
                gr, gm, bt = left.pop(0)
                sb.assign(k, gr, type("R", (), {"gammas": gm, "betas": bt})())
                running[k] = [gr, gm, bt, len(gm)]
        if not running:
            break
        sb.step()
        if step == 2:   # a running slot: its state after the layers it has run
            k, (gr, gm, bt, togo) = max(running.items(), key=lambda r: r[1][3])
            L = len(gm) - togo + 1
            if togo > 1:
                v = sb.copy_out(k, dtype).astype(np.complex128)
                _, _, want = _alone(N, gr, gm[:L], bt[:L], dtype)
                assert np.linalg.norm(v - want) / np.linalg.norm(want) < TOL[dtype], (k, L)
        done = []
        for k in list(running):
            running[k][3] -= 1
            if running[k][3] == 0:
                done.append((k, running.pop(k), sb.copy_out(k, dtype).astype(np.complex128), sb.slot_req[k]))
        while sb.poll():
            pass
        assert len(sb.collect()) == len(done)
        for k, (gr, gm, bt, _), v, req in done:
            e, n2, want = _alone(N, gr, gm, bt, dtype)
            assert np.linalg.norm(v - want) / np.linalg.norm(want) < TOL[dtype], (k, len(gm))
            assert req.expect == pytest.approx(e, rel=TOL[dtype])
            assert req.norm2 == pytest.approx(n2, abs=TOL[dtype])
    assert not left and not running
    sb.destroy()
    for gr in graphs:
        gr.destroy()
