"""The two-pass route of short runs (every duration first, then the propagation level by level) against the
walk of a configured shape and the oracle, bit for bit."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import dags as D
import oracle
from mc_dagprop_amd import capi
from mc_dagprop_amd.workloads import FlatDag, layered_vectorized, network_dists, seeded_network_dists

pytestmark = pytest.mark.gpu


def bits(a: np.ndarray) -> np.ndarray:
    return np.ascontiguousarray(a).view(np.uint64)


def two_pass(P: capi.Propagator, n: int, injected: bool = False) -> bool:
    yes = C.c_int32(0)
    capi.check(capi.lib().mcdp_debug_short_run(P.h, int(injected), n, C.byref(yes)))
    return bool(yes.value)


DAGS = {
    # 1-4 predecessors, every law of the network workload
    "layered": lambda: layered_vectorized(40, 30, 4, network_dists(), 8, 5),
    # stale reads, repeated targets and sources, shared links, gaps, edges outside the link table
    "edge_cases": lambda: D.continuous_dag(7, 400, max_delay=12.0, shared_links=True),
    # events of 20 and of 260 predecessors (more than an item holds inline), long-lived values
    "fan_in": lambda: D.long_lived_slots(3, fan_in=240),
    "chain": lambda: D.parity_long_chain(120),
    # levels of 300 events: 600 live values, more than LDS holds for 64 samples a workgroup
    "wide": lambda: layered_vectorized(6, 300, 4, seeded_network_dists(2), 8, 9),
}
# one sample; group sizes 1 | 2 at one workgroup per CU (256 | 257); a wave's edges; 64 a workgroup with a ragged last
COUNTS = [1, 2, 63, 64, 65, 256, 257, 1000, 9001]


@pytest.mark.parametrize("n", COUNTS)
@pytest.mark.parametrize("name", sorted(DAGS))
def test_two_pass_route_matches_walk_and_oracle(gpu, name: str, n: int) -> None:
    dag = DAGS[name]()
    seeds = np.arange(n, dtype=np.int32) * 17 - 4000
    A = capi.Propagator(dag)
    A.configure(16, 8, 1)
    B = capi.Propagator(dag)
    assert not two_pass(A, n)
    if n <= 1000:
        assert two_pass(B, n) and two_pass(B, n, injected=True)
    ra, da, ca = A.run_many(seeds)
    rb, db, cb = B.run_many(seeds)
    np.testing.assert_array_equal(bits(db), bits(da))
    np.testing.assert_array_equal(bits(rb), bits(ra))
    np.testing.assert_array_equal(cb, ca)
    dur = D.special_durations(np.random.default_rng(n), n, dag.link_count)
    ri, ci = A.propagate(dur)
    rj, cj = B.propagate(dur)
    np.testing.assert_array_equal(bits(rj), bits(ri))
    np.testing.assert_array_equal(cj, ci)
    pick = np.unique(np.r_[0:min(n, 40), max(0, n - 40):n])
    ro, co = oracle.OracleCtx(dag).propagate(dur[pick])
    np.testing.assert_array_equal(bits(rj[pick]), bits(ro))
    np.testing.assert_array_equal(cj[pick], co)


def test_two_pass_route_with_leading_dimension_and_without_causes(gpu) -> None:
    """Rows longer than the run, no cause output, and new times after the first run."""
    dag = DAGS["layered"]()
    n, ld = 130, 200
    seeds = np.arange(n, dtype=np.int32)
    P = capi.Propagator(dag)
    assert two_pass(P, n)
    sd = capi.DeviceBuffer.from_array(seeds)
    r = capi.DeviceBuffer.from_array(np.full((P.E, ld), -7.0))
    d = capi.DeviceBuffer.from_array(np.full((P.L, ld), -7.0))
    for shift in (0.0, 5.0):
        earliest = dag.earliest + shift
        P.set_times(earliest=earliest)
        P.run_many_device(sd, n, ld, r, d, None)
        capi.synchronize()
        Q = capi.Propagator(dag)
        Q.set_times(earliest=earliest)
        Q.configure(8, 4, 2)
        rq, dq, _ = Q.run_many(seeds)
        rr, dd = r.to_array(np.float64, (P.E, ld)), d.to_array(np.float64, (P.L, ld))
        np.testing.assert_array_equal(bits(rr[:, :n]), bits(rq.T))
        np.testing.assert_array_equal(bits(dd[:, :n]), bits(dq.T))
        assert (rr[:, n:] == -7.0).all() and (dd[:, n:] == -7.0).all()


@pytest.mark.parametrize("n", [1, 300])
def test_two_pass_statistics_match_rows(gpu, n: int) -> None:
    """run_stats of a short run (durations in the workspace, winner positions) equals the rows' statistics."""
    dag = DAGS["edge_cases"]()
    P = capi.Propagator(dag)
    assert two_pass(P, n)
    seeds = np.arange(n, dtype=np.int32) + 3
    mean, quant, counts = P.run_stats(seeds, (0.25, 0.5))
    Q = capi.Propagator(dag)
    Q.configure(16, 8, 2)
    m2, q2, c2 = Q.run_stats(seeds, (0.25, 0.5))
    np.testing.assert_array_equal(bits(mean), bits(m2))
    np.testing.assert_array_equal(bits(quant), bits(q2))
    np.testing.assert_array_equal(counts, c2)


@pytest.mark.parametrize("configured", [False, True])
def test_signed_zero_caps(gpu, configured: bool) -> None:
    """max_delay -0 makes caps of -0, where the smaller of -0 and +0 is not what the comparison keeps."""
    events = [(-0.0, 9.0, 0.0), (0.0, 9.0, 0.0), (-0.0, 9.0, 0.0), (-0.0, 9.0, 0.0)]
    acts = {(0, 1): (0, 0.0, 0), (0, 2): (1, 0.0, 0), (1, 3): (2, 0.0, 0), (2, 3): (3, 0.0, 0)}
    prec = [(1, [(0, 0)]), (2, [(0, 1)]), (3, [(1, 2), (2, 3)])]
    dag = FlatDag.from_lists(events, acts, prec, -0.0)
    vals = np.array([0.0, -0.0, 1.0, -1.0, np.nan])
    dur = np.stack(np.meshgrid(vals, vals, vals, vals), -1).reshape(-1, 4)
    P = capi.Propagator(dag)
    if configured:
        P.configure(4, 4, 2)
    r, c = P.propagate(dur)
    ro, co = oracle.OracleCtx(dag).propagate(dur)
    np.testing.assert_array_equal(bits(r), bits(ro))
    np.testing.assert_array_equal(c, co)


@pytest.mark.parametrize("ld_extra", [0, 5])
@pytest.mark.parametrize("n", [10000, 16384, 16385])
def test_halved_tiles_match(gpu, n: int, ld_extra: int) -> None:
    """Up to 64 samples per CU (16,384 on 256) a walk takes one-sample tiles where rows start on sectors: the
    bits of the configured shape, whole and split."""
    dag = layered_vectorized(8, 120, 4, network_dists(), 8, 11)
    ld = n + ld_extra
    seeds = capi.DeviceBuffer.from_array(np.arange(n, dtype=np.int32))
    out = []
    for configured in (False, True):
        P = capi.Propagator(dag)
        if configured:
            P.configure(16, 8, 2)
        r, d, c = (capi.DeviceBuffer(8 * P.E * ld), capi.DeviceBuffer(8 * P.L * ld), capi.DeviceBuffer(4 * P.E * ld))
        P.run_many_device(seeds, n, ld, r, d, c)
        capi.synchronize()
        res = [r.columns(np.float64, P.E, ld, 0, n), d.columns(np.float64, P.L, ld, 0, n),
               c.columns(np.int32, P.E, ld, 0, n)]
        P.run_many_device(seeds, n, ld, r, None, None)
        capi.synchronize()
        np.testing.assert_array_equal(bits(r.columns(np.float64, P.E, ld, 0, n)), bits(res[0]))
        out.append(res)
    np.testing.assert_array_equal(bits(out[0][0]), bits(out[1][0]))
    np.testing.assert_array_equal(bits(out[0][1]), bits(out[1][1]))
    np.testing.assert_array_equal(out[0][2], out[1][2])
