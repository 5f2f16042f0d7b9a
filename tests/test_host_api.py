"""The host side of the library on the CPU (tests/host_api.cpp): fq_api.cpp compiled
against host memory and launchers that check what they are given."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="session")
def host_api(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_api") / "host_api")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                           f"-I{ROOT}/include", f"-I{ROOT}/for-qaoa_amd/csrc", f"{ROOT}/tests/host_api.cpp",
                           "-o", exe])

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        return dict((k, int(v)) for k, v in re.findall(r"(\w+) (-?\d+)", r.stdout))

    return run


@pytest.mark.parametrize("call,N,dtype,P,small", [
    # 64 plans are kept; the <C> plans that fill the cache are smaller than the calls'
    ("run", 22, 0, 3, 62), ("run", 22, 0, 3, 63), ("run", 24, 0, 5, 63), ("run", 23, 1, 3, 63), ("run", 28, 1, 2, 63),
    ("z2", 24, 0, 3, 63), ("z2", 28, 1, 3, 62), ("run", 12, 0, 3, 63), ("run", 20, 1, 3, 64),
    ("backward", 22, 0, 3, 62), ("backward", 26, 1, 2, 62), ("backward", 24, 0, 3, 63),
    ("slab", 16, 0, 3, 63), ("slab_z2", 23, 1, 3, 62), ("slab_z2", 24, 0, 3, 63), ("slab", 25, 1, 3, 63),
    # plans of equal size: the least recently used ones are replaced throughout
    ("run", 16, 0, 3, 70), ("slab", 20, 1, 3, 70), ("slab_z2", 8, 0, 3, 70),
])
def test_plans_stay_until_they_are_read(host_api, call, N, dtype, P, small):
    """A full plan cache: no plan that a call has looked up is replaced before the
    launches that read it, and the cache stays bounded."""
    r = host_api("plans", call, N, dtype, P, small)
    assert r["checked"] > small and r["wrong"] == 0
    assert r["cached"] <= 64 + 5   # (a call's own plans at most beyond the limit)


@pytest.mark.parametrize("N,dtype,schedule,depths", [
    # one launch of all layers; all tables at once, in a first buffer that holds them and
    # in one that does not; a table for each pass, with and without chunks
    (12, 0, 1, (4, 64, 70)), (16, 0, 1, (4, 30, 64)), (20, 1, 1, (4, 30, 64)), (22, 0, 1, (4, 40, 64)),
    (22, 0, 2, (5, 41, 64)), (25, 1, 1, (4, 9, 20)), (28, 1, 1, (3, 6, 9)), (26, 0, 2, (5, 7, 8)),
    # a first run of one layer makes the room of one table
    (12, 0, 1, (1, 3, 64)), (11, 1, 2, (1, 66, 2)), (16, 0, 1, (1, 3, 64)), (22, 1, 1, (1, 4, 2)),
])
def test_captured_runs_keep_their_tables(host_api, N, dtype, schedule, depths):
    """A run that is captured, deeper than the one before it, allocates nothing, and the
    tables its launches read outlive what grows after it, as long as the state."""
    r = host_api("capture", N, dtype, schedule, *depths)
    assert r["checked"] > 0 and r["wrong"] == 0
    assert r["kept"] == 0


@pytest.mark.parametrize("N,dtype,schedule", [(14, 0, 1), (16, 1, 2), (23, 1, 2), (25, 0, 2)])
def test_open_layer_takes_a_change_once(host_api, N, dtype, schedule):
    """A step that fails once the open layer has the new weights does not add the
    difference again when it is called again."""
    r = host_api("reopen", N, dtype, schedule)
    assert r["failed"] == 1 and r["reopened"] == 1 and r["again"] == 1


@pytest.mark.parametrize("N,dtype,schedule", [
    # general, packed, one by one; the half states of 24 qubits in between
    (3, 0, 2), (9, 0, 1), (10, 0, 1), (10, 1, 2), (11, 1, 2), (21, 0, 2), (22, 0, 2), (22, 1, 1), (23, 1, 2), (24, 1, 2),
    (24, 0, 1), (25, 0, 1), (25, 1, 2), (30, 1, 2),
])
@pytest.mark.parametrize("P", [1, 2, 5])
def test_slab_passes_are_those_launched(host_api, N, dtype, schedule, P):
    r = host_api("passes", N, dtype, schedule, P)
    assert r["launched"] == r["told"] > 0


def test_serving_floor_counts_the_passes_that_run():
    # packed slots of N=16 run 1 + P passes of a half state, not 2 P
    from forqaoa.serve import Request, Stream, bytes_floor
    r = Request(0, 16, 5, 0, [0.1] * 5, [0.2] * 5)
    S = (1 << 15) * 8
    assert bytes_floor(Stream({}, [r]), [r], "c64", "z2") == S * (2 * 6 - 1) + S


def test_default_plans_cover_every_layer(host_api):
    """The plans that fq_run and the gradient run without tuning knobs, for every N, both
    types, the full and the half state."""
    r = host_api("cover", 1, 36)
    assert r["checked"] > 10000 and r["wrong"] == 0


@pytest.mark.parametrize("call,N,dtype", [("run", 11, 0), ("run", 14, 0), ("z2", 25, 1), ("run", 27, 0),
                                          ("backward", 14, 1), ("backward", 25, 0)])
def test_deep_runs_stay_small(host_api, call, N, dtype):
    """A run keeps some tens of bytes of host memory for each layer (the list of its
    passes, a gradient's sums), not the launch arguments of all passes."""
    assert host_api("deep", call, N, dtype, 4000)["bytes_per_layer"] < 256


@pytest.mark.parametrize("N,dtype,schedule,P,kib", [(12, 0, 1, 30, 64), (11, 1, 2, 67, 64), (16, 0, 1, 30, 64),
                                                    (21, 1, 2, 30, 256)])
def test_runs_without_memory_for_all_tables(host_api, N, dtype, schedule, P, kib):
    """A table at a time, as before all of a run's tables were made at once."""
    r = host_api("nomem", N, dtype, schedule, P, kib)
    assert r["checked"] == P and r["wrong"] == 0


@pytest.mark.parametrize("N,dtype,schedule", [(12, 0, 1), (14, 0, 1), (16, 1, 2), (9, 1, 1)])
def test_plans_first_made_under_capture(host_api, N, dtype, schedule):
    """Their upload happens on each replay, so only the captured run may count on them."""
    r = host_api("newplan", N, dtype, schedule, 3)
    assert r["checked"] > 0 and r["nodes"] > 0 and r["wrong"] == 0


@pytest.mark.parametrize("N,dtype,P", [(22, 0, 2), (24, 0, 1)])
def test_captured_plans_outlive_a_drop_of_the_cache(host_api, N, dtype, P):
    """A call whose plans are larger than all 64 cached ones drops those, but not the memory
    that a captured run's graph uploads its plans to and reads them from on each replay."""
    r = host_api("dropped", N, dtype, P)
    assert r["drops"] > 0 and r["nodes"] > 0 and r["wrong"] == 0


@pytest.mark.parametrize("call,N,dtype", [
    # packed slots; slots one by one in two and three passes, in layer order
    ("slab", 14, 1), ("slab_z2", 16, 1), ("slab_z2", 20, 0), ("slab_z2", 22, 1), ("slab_z2", 23, 1), ("slab", 25, 1),
    ("slab_z2", 25, 1), ("slab_z2", 26, 0), ("slab", 29, 1),
])
@pytest.mark.parametrize("P", [1, 2, 3, 6])
def test_factors_of_slots_go_into_the_cost_phases(host_api, call, N, dtype, P):
    """No factor is multiplied into all amplitudes alike (rounded to FP32 it would change the
    norm), and their product is that of the layers' RX: 1e-12, some N P roundings in FP64."""
    r = host_api("factors", call, N, dtype, P)
    assert r["common"] == 0 and r["off"] == 0


@pytest.mark.parametrize("N,dtype,K", [(8, 1, 16), (16, 1, 32), (12, 0, 4)])
def test_plans_of_slots_that_enter_together_go_in_one_copy(host_api, N, dtype, K):
    """And the step's parameters in another."""
    r = host_api("copies", N, dtype, K)
    assert r["copies"] == 2 and r["checked"] > K and r["wrong"] == 0
