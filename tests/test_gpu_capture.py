"""Runs captured into HIP graphs after a first run of another size or route, bit for bit against eager runs.

A propagator's plans reach the device when a run first needs them, so a captured run may need one that the run
before it did not; and the two launches of a short run are captured as they are."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from mc_dagprop_amd import capi
from mc_dagprop_amd.workloads import layered_network, layered_vectorized, network_dists, seeded_network_dists

pytestmark = pytest.mark.gpu


def two_pass(P: capi.Propagator, n: int) -> bool:
    yes = C.c_int32(0)
    capi.check(capi.lib().mcdp_debug_short_run(P.h, 0, n, C.byref(yes)))
    return bool(yes.value)


class Run:
    """Device buffers of a sampled run of n samples."""

    def __init__(self, P: capi.Propagator, n: int, durations: bool = True) -> None:
        self.P, self.n = P, n
        self.seeds = capi.DeviceBuffer.from_array(np.arange(n, dtype=np.int32) * 5 - 9)
        self.real, self.cause = capi.DeviceBuffer(8 * P.E * n), capi.DeviceBuffer(4 * P.E * n)
        self.dur = capi.DeviceBuffer(8 * P.L * n) if durations else None

    def launch(self, stream) -> None:
        self.P.run_many_device(self.seeds, self.n, self.n, self.real, self.dur, self.cause, stream)

    def overwrite(self) -> None:
        for b in (self.real, self.cause, self.dur):
            if b is not None:
                capi.check(capi.lib().mcdp_memset(b.ptr, 0xFF, b.nbytes))

    def read(self) -> list[np.ndarray]:
        capi.synchronize()
        out = [self.real.to_array(np.uint64, (self.P.E, self.n)), self.cause.to_array(np.int32, (self.P.E, self.n))]
        return out + ([self.dur.to_array(np.uint64, (self.P.L, self.n))] if self.dur is not None else [])


class Stream:
    def __enter__(self):
        self.s = C.c_void_p(0)
        capi.check(capi.lib().mcdp_stream_create(C.byref(self.s)))
        return self.s

    def __exit__(self, *exc) -> None:
        capi.check(capi.lib().mcdp_stream_destroy(self.s))


DAGS = {
    "layered": lambda: layered_vectorized(20, 30, 4, network_dists(), 8, 5),
    # 600 live values: more than 64 KB of LDS in the second launch of a short run
    "wide": lambda: layered_vectorized(6, 300, 4, seeded_network_dists(2), 8, 9),
}


@pytest.mark.parametrize("first,n,durations", [(10, 40_000, True), (10, 300, False), (40_000, 300, True), (300, 300, True)])
@pytest.mark.parametrize("name", sorted(DAGS))
def test_capture_after_a_first_run(gpu, name: str, first: int, n: int, durations: bool) -> None:
    dag = DAGS[name]()
    P, Q, other = capi.Propagator(dag), capi.Propagator(dag), capi.Propagator(layered_network(layers=12))
    assert two_pass(P, 10) and two_pass(P, 300) and not two_pass(P, 40_000)
    want = Run(Q, n, durations)
    want.launch(None)
    expected = want.read()
    warm = Run(P, first)
    warm.launch(None)
    capi.synchronize()
    got, graph = Run(P, n, durations), C.c_void_p(0)
    with Stream() as stream:
        capi.check(capi.lib().mcdp_graph_capture_begin(stream))
        got.launch(stream)
        capi.check(capi.lib().mcdp_graph_capture_end(stream, C.byref(graph)))
        for rep in range(3):
            got.overwrite()
            other.run_many(np.arange(300))
            capi.check(capi.lib().mcdp_graph_launch(graph, stream))
            capi.synchronize(stream)
            for a, b in zip(got.read(), expected):
                np.testing.assert_array_equal(a, b, err_msg=f"replay {rep}")
        capi.check(capi.lib().mcdp_graph_destroy(graph))
        # eager runs of either route go on as before
        short = Run(P, 10)
        for again in (got, short):
            again.overwrite()
            again.launch(stream)
        for a, b in zip(got.read(), expected):
            np.testing.assert_array_equal(a, b)


def test_short_run_beside_a_capture(gpu) -> None:
    """A short run on one stream while another stream is being captured, on a propagator that has only walked."""
    dag = DAGS["layered"]()
    P, Q = capi.Propagator(dag), capi.Propagator(dag)
    long_run, small = Run(Q, 40_000), Run(P, 64)
    walk = Run(P, 40_000)
    walk.launch(None)
    long_run.launch(None)
    expected, graph = long_run.read(), C.c_void_p(0)
    with Stream() as stream, Stream() as beside:
        capi.check(capi.lib().mcdp_graph_capture_begin(stream))
        long_run.launch(stream)
        small.launch(beside)
        capi.check(capi.lib().mcdp_graph_capture_end(stream, C.byref(graph)))
        long_run.overwrite()
        capi.check(capi.lib().mcdp_graph_launch(graph, stream))
        capi.synchronize(stream)
        for a, b in zip(long_run.read(), expected):
            np.testing.assert_array_equal(a, b)
        capi.check(capi.lib().mcdp_graph_destroy(graph))
    for a, b in zip(small.read(), expected):
        np.testing.assert_array_equal(a, b[:, :64])
