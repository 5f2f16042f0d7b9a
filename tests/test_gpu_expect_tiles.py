"""<C> of states whose tiles' sums are added up on the host (up to 256 tiles, N = 20) and of
the smallest ones that take a second launch, against the allocation-free entry point, which
always takes one: the same order of additions, equal to the last bit."""
import pytest

import test_gpu_lanes as lanes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["c128", "c64"])
@pytest.mark.parametrize("N", [14, 16, 18, 19, 20])
def test_expect_of_few_tiles(N, dtype):
    lanes.test_expect_equals_two_launches(N, dtype)
