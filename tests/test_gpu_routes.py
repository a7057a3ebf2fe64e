"""The routes a run can take, each shown to be the one that ran, bit for bit against another."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import dags as D
from mc_dagprop_amd import capi
from mc_dagprop_amd.workloads import FlatDag, layered_network, layered_small, layered_vectorized, network_dists

pytestmark = pytest.mark.gpu

TWO_PASS, TILES, ONE_SAMPLE, OVERLAPPING, WIDE, GRAPH = 1, 2, 4, 8, 16, 32


def bits(a: np.ndarray) -> np.ndarray:
    return np.ascontiguousarray(a).view(np.uint64)


def route(P: capi.Propagator) -> int:
    r = C.c_int32(-1)
    capi.check(capi.lib().mcdp_debug_last_route(P.h, C.byref(r)))
    return r.value


def two_pass_mode(P: capi.Propagator, mode: int) -> None:
    capi.check(capi.lib().mcdp_debug_two_pass_mode(P.h, mode))


def run_device(P: capi.Propagator, n: int, ld: int, durations: bool = True) -> list[np.ndarray]:
    seeds = capi.DeviceBuffer.from_array(np.arange(n, dtype=np.int32) * 3 + 1)
    r, c = capi.DeviceBuffer(8 * P.E * ld), capi.DeviceBuffer(4 * P.E * ld)
    d = capi.DeviceBuffer(8 * P.L * ld) if durations else None
    P.run_many_device(seeds, n, ld, r, d, c)
    capi.synchronize()
    out = [r.columns(np.uint64, P.E, ld, 0, n), c.columns(np.int32, P.E, ld, 0, n)]
    return out + ([d.columns(np.uint64, P.L, ld, 0, n)] if durations else [])


TWO_PASS_DAGS = {
    "layered": lambda: layered_vectorized(40, 30, 4, network_dists(), 8, 5),
    "edge_cases": lambda: D.continuous_dag(7, 400, max_delay=12.0, shared_links=True),
    "fan_in": lambda: D.long_lived_slots(3, fan_in=240),
}


@pytest.mark.parametrize("n", [150, 300, 700, 1500, 3000, 6001, 12_000, 20_011])
@pytest.mark.parametrize("name", sorted(TWO_PASS_DAGS))
def test_two_passes_of_every_group_size(gpu, name: str, n: int) -> None:
    """1 to 64 samples a workgroup (256 CUs: the doubled sample counts), and more workgroups than CUs."""
    dag = TWO_PASS_DAGS[name]()
    A, B = capi.Propagator(dag), capi.Propagator(dag)
    two_pass_mode(A, 2)
    two_pass_mode(B, 1)
    for a, b in zip(run_device(A, n, n), run_device(B, n, n)):
        np.testing.assert_array_equal(b, a)
    assert route(B) == TWO_PASS and not route(A) & TWO_PASS
    dur = D.special_durations(np.random.default_rng(n), n, dag.link_count)
    ra, ca = A.propagate(dur)
    rb, cb = B.propagate(dur)
    assert route(B) == TWO_PASS and not route(A) & TWO_PASS
    np.testing.assert_array_equal(bits(rb), bits(ra))
    np.testing.assert_array_equal(cb, ca)


@pytest.mark.parametrize("n", [24_577, 30_721, 32_767, 45_002])
@pytest.mark.parametrize("width,shape", [(60, (16, 4, 2)), (100, (16, 8, 2))])
def test_overlapping_tiles_of_both_sizes(gpu, width: int, shape, n: int) -> None:
    """Rows off the cache sectors, for plans of 4 and of 8 events per wave, against rows on them."""
    P = capi.Propagator(layered_vectorized(6, width, 4, network_dists(), 8, 77000))
    P.configure(*shape)
    want = run_device(P, n, (n + 15) // 16 * 16)
    assert not route(P) & OVERLAPPING
    for a, b in zip(run_device(P, n, n + (n + 1) % 2), want):
        np.testing.assert_array_equal(a, b)
    assert route(P) & OVERLAPPING


@pytest.mark.parametrize("n", [10_000, 16_384])
@pytest.mark.parametrize("durations", [True, False])
def test_one_sample_tiles(gpu, durations: bool, n: int) -> None:
    dag = layered_vectorized(8, 120, 4, network_dists(), 8, 11)
    P, Q = capi.Propagator(dag), capi.Propagator(dag)
    two_pass_mode(P, 2)
    Q.configure(16, 8, 2)
    for a, b in zip(run_device(P, n, n, durations), run_device(Q, n, n, durations)):
        np.testing.assert_array_equal(a, b)
    assert route(P) == ONE_SAMPLE and route(Q) == TILES


def replayed(P: capi.Propagator, want, call) -> None:
    got = call()
    assert route(P) == GRAPH
    for a, b in zip(got, want):
        np.testing.assert_array_equal(bits(a) if a.dtype == np.float64 else a, bits(b) if b.dtype == np.float64 else b)


@pytest.mark.parametrize("name", ["network_slice", "long_chain"])
def test_short_walks_replay_a_graph(gpu, name: str) -> None:
    """Short host runs that walk: from the second call with a sample count on, a graph of the walk's launches is
    replayed, with other work between the replays; new times are not hidden by it."""
    dag = layered_network(layers=40) if name == "network_slice" else D.parity_long_chain(99)
    P, Q, other = capi.Propagator(dag), capi.Propagator(dag), capi.Propagator(layered_small())
    two_pass_mode(P, 2)
    seeds = np.arange(6, dtype=np.int32) * 13 + 5
    want = Q.run_many(seeds)
    assert route(Q) == TWO_PASS
    P.run_many(seeds)
    assert route(P) & (WIDE | ONE_SAMPLE | TILES)
    for k in range(4):
        replayed(P, want, lambda: P.run_many(seeds))
        other.run_many(np.arange(50 + k))
        capi.synchronize()
    P.propagate(want[1])
    assert route(P) != GRAPH
    for _ in range(3):
        replayed(P, (want[0], want[2]), lambda: P.propagate(want[1]))
    moved = FlatDag(**{**dag.__dict__})
    moved.earliest = P.get_times()[1] + 7.0
    P.set_times(earliest=moved.earliest)
    want = capi.Propagator(moved).run_many(seeds)
    got = P.run_many(seeds)
    assert route(P) != GRAPH
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
    for _ in range(2):
        replayed(P, want, lambda: P.run_many(seeds))
