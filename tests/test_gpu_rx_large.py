"""RX on qubits below C of complex64 states beyond the memory-side cache, whose tiles hold
2^11 amplitudes at least whatever C is, and the largest size below: against RX in numpy
on one factor of a product state.

Tolerance: one FMA per component and gate on a unit-norm state, under 20 eps (RX(2.6),
beyond the butterfly's first branch, as two): 3e-5 with a margin.
"""
import numpy as np
import pytest

from forqaoa import State

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,C,targets", [
    (26, 10, range(10)), (26, 9, range(9)), (26, 1, range(1)), (26, 10, (0, 3, 9)), (26, 11, range(11)),
    (27, 5, range(1, 5)), (25, 10, range(10)),
])
@pytest.mark.parametrize("beta", [0.7, 2.6])
def test_rx_below_c(N, C, targets, beta):
    targets = list(targets)
    print(f"RX({beta}) on {targets} of N={N} complex64, C={C}", flush=True)
    rng = np.random.default_rng(N + C)
    a = rng.normal(size=1 << 12) + 1j * rng.normal(size=1 << 12)
    b = rng.normal(size=1 << (N - 12)) + 1j * rng.normal(size=1 << (N - 12))
    a /= np.linalg.norm(a)
    b /= np.linalg.norm(b)
    st = State(N, C=C, dtype="c64")
    st.copy_in((b[:, None] * a[None, :]).reshape(-1).astype(np.complex64))
    st.multi_rx(targets, beta)
    got = st.copy_out().reshape(-1, 1 << 12)
    st.destroy()
    c, s = np.cos(beta / 2), -1j * np.sin(beta / 2)
    for q in targets:
        x = a.reshape(-1, 2, 1 << q)
        a = np.stack([c * x[:, 0] + s * x[:, 1], s * x[:, 0] + c * x[:, 1]], axis=1).reshape(-1)
    err = 0.0
    for i in range(0, 1 << (N - 12), 1024):
        d = got[i:i + 1024] - b[i:i + 1024, None] * a[None, :]
        err += float(np.sum(np.abs(d) ** 2))
    assert np.sqrt(err) < 3e-5
