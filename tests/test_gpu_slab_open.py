"""A running slot's amplitudes while its last layer is open: that layer's cost pass has taken
the RX factors of the passes that are still to come, which the copy-out must not show."""
import numpy as np
import pytest

from forqaoa import Graph, State
from forqaoa import graphs as G
from forqaoa.serve import Slab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dtype,schedule", [(14, "c128", "z2"), (16, "c64", "fused"), (23, "c64", "z2"), (25, "c64", "fused"),
                                              (24, "c128", "fused")])
def test_copy_out_with_the_last_layer_open(N, dtype, schedule):
    """Against a run of as many layers, within (N + 2) P roundings of a unit-norm state: 1e-12
    and 1e-5 with a margin."""
    print(f"copy-out N={N} {dtype} {schedule}", flush=True)
    gr = Graph(N, G.gnp(N, 0.4, 9400 + N, "uniform"))
    sb, st = Slab(N, 1, dtype, schedule), State(N, C=min(N, 12), dtype=dtype)
    P = 4
    g, b = G.angles(P, 9500 + N)
    b[3] = 2.9   # the butterfly's other branch
    sb.assign(0, gr, type("R", (), {"gammas": g, "betas": b})())
    for p in range(1, P):
        sb.step()
        while sb.poll():
            pass
        got = sb.copy_out(0, dtype).astype(np.complex128)
        st.run(gr, g[:p], b[:p], "fused")
        want = st.copy_out().astype(np.complex128)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) < (1e-12 if dtype == "c128" else 1e-5), p
    sb.destroy()
    st.destroy()
    gr.destroy()
