"""Workspaces of more than 4 GiB are kept between calls and shared by the propagators of a process: results do
not depend on what a workspace held before, from several threads, and the memory goes back with its propagators."""

from __future__ import annotations

import ctypes
import gc
import threading

import numpy as np
import pytest

from mc_dagprop_amd import capi
from mc_dagprop_amd.workloads import layered_vectorized, network_dists

pytestmark = pytest.mark.gpu


def mem_info() -> tuple[int, int]:
    """Free and total device memory, asked of the HIP runtime that the library itself uses."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert capi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value, total.value


def test_large_workspaces_are_shared_and_given_back(gpu) -> None:
    n = 27000  # rows of 20,000 events: 4.9e9 bytes of statistics workspace, 1.7e10 of a gradient's
    dags = [layered_vectorized(200, 100, 4, network_dists(), 8, s) for s in (1, 2)]
    seeds = [np.arange(n, dtype=np.int32) + 10 * k for k in range(2)]
    w = np.linspace(0.5, 2.0, dags[0].n_events)
    props = [capi.Propagator(d) for d in dags]
    for p in props:
        p.run_stats(seeds[0][:8])  # plans resident
    free0 = mem_info()[0]
    first = [p.run_stats(s) for p, s in zip(props, seeds)]
    grads = [p.gradient(s, w) for p, s in zip(props, seeds)]
    again = [p.run_stats(s) for p, s in zip(props, seeds)]  # in workspaces the gradients used
    for a, b in zip(first, again):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)
    got: dict = {}

    def work(k: int) -> None:
        got[k] = [props[k].run_stats(seeds[k]) for _ in range(3)] + [props[k].gradient(seeds[k], w)]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        for r in got[k][:3]:
            for x, y in zip(first[k], r):
                np.testing.assert_array_equal(x, y)
        assert got[k][3][0] == grads[k][0]
        np.testing.assert_array_equal(got[k][3][1], grads[k][1])
        np.testing.assert_array_equal(got[k][3][2], grads[k][2])
    held = free0 - mem_info()[0]
    total = mem_info()[1]
    assert held < total / 8 + (6 << 30)  # the pool's bound, the reverse plans and partial rows
    del props, p
    gc.collect()
    assert mem_info()[0] > free0 - (1 << 30)
