"""Qubit exchanges of states beyond the memory-side cache (complex128 from N=25, complex64
from N=26, whose tiles also load a unit ahead): fewer work-groups than CUs, bitwise
against the axis permutation in numpy."""
import numpy as np
import pytest

import refmath as R
from forqaoa import State

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dtype,out,inn,k", [
    (26, "c64", 0, 13, 13), (26, "c64", 0, 12, 10), (26, "c64", 0, 25, 1), (26, "c64", 3, 14, 5), (26, "c64", 20, 24, 2),
    (27, "c64", 0, 14, 8), (25, "c128", 0, 12, 12), (25, "c128", 0, 13, 3), (25, "c128", 4, 22, 2), (26, "c128", 11, 20, 6),
])
def test_exchange_large(N, dtype, out, inn, k):
    print(f"exchange N={N} {dtype} [{out},+{k}) [{inn},+{k})", flush=True)
    i = np.arange(1 << N)   # every amplitude its own value, exact in FP32
    v = (i % 8192 + 1j * (i // 8192)).astype(np.complex128 if dtype == "c128" else np.complex64)
    st = State(N, C=10, dtype=dtype)
    st.copy_in(v)
    st.swap_conti(out, inn, k)
    got = st.copy_out()
    st.destroy()
    np.testing.assert_array_equal(got, R.axis_swap_blocks(v, N, out, inn, k))
