"""A slab of as many slots as a grid's second dimension allows (65,536): a step that opens two
layers in each makes twice as many phase tables, in several launches.

The passes are those of a slab of 4 slots with the same requests: equal to the last bit.
"""
import pytest

from forqaoa import Graph
from forqaoa import graphs as G
from forqaoa.serve import Slab

pytestmark = pytest.mark.gpu


def _run(K, N, graphs, angles):
    sb = Slab(N, K, "c64", "z2")
    reqs = []
    for k in range(K):
        g, b = angles[k % 4]
        reqs.append(type("R", (), {"gammas": g, "betas": b})())
        sb.assign(k, graphs[k % 4], reqs[-1])
    for _ in range(2):
        sb.step()
    while sb.poll():
        pass
    assert len(sb.collect()) == K
    sb.destroy()
    return [(r.expect, r.norm2) for r in reqs]


def test_as_many_slots_as_a_grid_takes():
    N, K = 11, 65536
    print(f"slab of {K} slots, N={N}", flush=True)
    graphs = [Graph(N, G.gnp(N, 0.5, 9600 + i, "uniform")) for i in range(4)]
    angles = [G.angles(2, 9700 + i) for i in range(4)]
    want = _run(4, N, graphs, angles)
    got = _run(K, N, graphs, angles)
    assert all(got[k] == want[k % 4] for k in range(K))
    for g in graphs:
        g.destroy()
