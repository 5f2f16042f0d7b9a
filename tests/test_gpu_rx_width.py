"""RX in tiles of the width that its number of targets takes: every width, on each side of
the sizes at which it changes, targets at the top, in the middle and apart, and few
targets of a wide chunk.  Against RX in numpy on the two factors of a product state.

Tolerance: one FMA per component and gate on a unit-norm state, under 20 eps (RX(2.6),
beyond the butterfly's first branch, as two): 3e-5 and 1e-13 with a margin.
"""
import numpy as np
import pytest

from forqaoa import State

pytestmark = pytest.mark.gpu

TOL = {"c128": 1e-13, "c64": 3e-5}


def _rx(v, targets, beta):
    c, s = np.cos(beta / 2), -1j * np.sin(beta / 2)
    for q in targets:
        x = v.reshape(-1, 2, 1 << q)
        v = np.stack([c * x[:, 0] + s * x[:, 1], s * x[:, 0] + c * x[:, 1]], axis=1).reshape(-1)
    return v


@pytest.mark.parametrize("N,dtype,C,counts", [
    # 16 MiB, from 32 MiB on, 256 MiB, 512 MiB
    (21, "c64", 10, (1, 5)), (22, "c64", 10, (1, 2, 3, 4, 5, 6)), (25, "c64", 10, (5, 6, 7)), (26, "c64", 10, (1, 5, 6)),
    (20, "c128", 10, (4, 5)), (21, "c128", 10, (1, 3, 4, 5, 6)), (24, "c128", 10, (5, 6, 7)), (25, "c128", 10, (1, 2, 3, 5, 6)),
    # chunks: narrower tiles than C in complex64, the whole of a small state
    (14, "c64", 13, ()), (22, "c64", 14, ()), (11, "c64", 10, ()), (10, "c64", 10, ()), (15, "c64", 9, ()), (15, "c128", 13, ()),
])
@pytest.mark.parametrize("beta", [0.7, 2.6])
def test_rx_by_number_of_targets(N, dtype, C, counts, beta):
    print(f"RX({beta}) N={N} {dtype} C={C} {counts}", flush=True)
    rng = np.random.default_rng(N + C)
    k = N // 2
    a, b = (rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n) for n in (k, N - k))
    a, b = a / np.linalg.norm(a), b / np.linalg.norm(b)
    sets = [s for n in counts for s in (range(N - n, N), range(C + 1, C + 1 + n), range(N - 1 - 2 * (n - 1), N, 2))]
    if not counts:
        sets = [[0], [C - 1], range(min(5, C)), range(C), [0, C // 2]]
    st = State(N, C=C, dtype=dtype)
    for targets in sets:
        targets = sorted(targets)
        st.copy_in((b[:, None] * a[None, :]).reshape(-1).astype(np.complex128 if dtype == "c128" else np.complex64))
        st.multi_rx(targets, beta)
        got = st.copy_out().reshape(1 << (N - k), 1 << k)
        x = _rx(a, [q for q in targets if q < k], beta)
        y = _rx(b, [q - k for q in targets if q >= k], beta)
        err = 0.0
        for i in range(0, 1 << (N - k), 256):
            err += float(np.sum(np.abs(got[i:i + 256] - y[i:i + 256, None] * x[None, :]) ** 2))
        assert np.sqrt(err) < TOL[dtype], targets
    st.destroy()
