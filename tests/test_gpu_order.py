"""Strided passes with runs of 128 B on states beyond the memory-side cache take
their tiles in another order (MixArgs::by_xcd): the smallest such states, RX on
as many top qubits as one pass takes, and on fewer, against RX in numpy.

Tolerance: one FMA per component and gate on a unit-norm state, under 20 eps:
1e-13 and 3e-5 with a margin, as for the other tile passes.
"""
import numpy as np
import pytest

from forqaoa import State

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dtype,k", [(25, "c128", 10), (25, "c128", 3), (26, "c64", 10), (26, "c64", 1)])
def test_rx_on_top_qubits(N, dtype, k):
    print(f"RX on the top {k} qubits of N={N} {dtype}", flush=True)
    rng = np.random.default_rng(N + k)
    # a few products of random factors: every amplitude its own value, made cheaply
    a = rng.normal(size=1 << 12) + 1j * rng.normal(size=1 << 12)
    b = rng.normal(size=1 << (N - 12)) + 1j * rng.normal(size=1 << (N - 12))
    v = (b[:, None] * a[None, :]).reshape(-1)
    v /= np.linalg.norm(v)
    st = State(N, C=12, dtype=dtype)
    st.copy_in(v.astype(st.np_dtype))
    beta = 0.7
    st.multi_rx(list(range(N - k, N)), beta)
    got = st.copy_out()
    st.destroy()
    # RX acts on b's factor only (the top qubits)
    c, s = np.cos(beta / 2), -1j * np.sin(beta / 2)
    w = b / (np.linalg.norm(a) * np.linalg.norm(b))
    for q in range(N - 12 - k, N - 12):
        x = w.reshape(-1, 2, 1 << q).copy()
        w = np.stack([c * x[:, 0] + s * x[:, 1], s * x[:, 0] + c * x[:, 1]], axis=1).reshape(-1)
    err = 0.0
    for i in range(0, 1 << (N - 12), 1024):
        d = got.reshape(-1, 1 << 12)[i:i + 1024] - w[i:i + 1024, None] * a[None, :]
        err += float(np.sum(np.abs(d) ** 2))
    assert np.sqrt(err) < {"c128": 1e-13, "c64": 3e-5}[dtype]
