"""Tile order by XCD (MixArgs::by_xcd) of strided passes with 128-byte runs, which starts
at states of 2 GiB: RX on the top qubits of the smallest such states (test_gpu_order has
the smaller ones, in order)."""
import pytest

import test_gpu_order as order

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dtype,k", [(27, "c128", 10), (28, "c64", 10), (28, "c64", 3)])
def test_rx_on_top_qubits_by_xcd(N, dtype, k):
    order.test_rx_on_top_qubits(N, dtype, k)
