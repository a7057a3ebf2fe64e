"""Sampled runs whose rows start off the cache sectors against the same run in aligned rows, bit for bit.

Overlapping tiles store each row from its own first whole sector: every row alignment, base pointers
off the sectors, and sample counts at the edges of a tile, of a round and of its remainder.  What lies
between the rows' last sample and ld stays as it was.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from mc_dagprop_amd import capi
from mc_dagprop_amd import workloads as wl

pytestmark = pytest.mark.gpu

ROUND = 256 * 120  # samples of one overlapping tile on each CU


class Rows:
    """An array of rows with `first` elements before it, filled with a value no result takes."""

    def __init__(self, rows: int, ld: int, dtype: torch.dtype, first: int) -> None:
        self.all = torch.full((first + rows * ld,), -77, dtype=dtype, device="cuda")
        self.view = self.all[first:].view(rows, ld)
        self.ptr = ctypes.c_void_p(self.view.data_ptr())


@pytest.fixture(scope="module")
def propagator():
    dag = wl.layered_vectorized(14, 100, 4, wl.network_dists(), 8, 77000)
    return capi.Propagator(dag)


@pytest.mark.parametrize(
    "n,pad,first",
    [(24_577, 0, 0), (27_005, 2, 1), (ROUND - 1, 0, 0), (ROUND, 3, 0), (ROUND + 1, 0, 3), (ROUND + 9, 4, 0),
     (32_767, 0, 0), (45_002, 1, 5), (2 * ROUND + 8, 5, 7), (2 * ROUND + 5003, 0, 2)],
)
def test_ragged_rows_equal_aligned_rows(gpu, propagator, n: int, pad: int, first: int) -> None:
    P = propagator
    seeds = Rows(1, n, torch.int32, 0)
    seeds.view[0] = torch.arange(n, dtype=torch.int32) * 3 + 1

    def run(ld: int, first: int) -> list[Rows]:
        out = [Rows(P.E, ld, torch.float64, first), Rows(P.L, ld, torch.float64, first), Rows(P.E, ld, torch.int32, first)]
        P.run_many_device(seeds, n, ld, *out)
        torch.cuda.synchronize()
        return out

    want = run((n + 15) // 16 * 16, 0)
    for got, ref in zip(run(n + pad, first), want):
        assert torch.equal(got.view[:, :n].contiguous().view(torch.int32), ref.view[:, :n].contiguous().view(torch.int32))
        assert bool((got.view[:, n:] == -77).all()) and bool((got.all[:first] == -77).all())


def test_without_causes(gpu, propagator) -> None:
    P, n = propagator, 33_001
    seeds = Rows(1, n, torch.int32, 0)
    seeds.view[0] = torch.arange(n, dtype=torch.int32)
    one = [Rows(P.E, n, torch.float64, 0), Rows(P.L, n, torch.float64, 0), Rows(P.E, n, torch.int32, 0)]
    two = [Rows(P.E, n, torch.float64, 0), Rows(P.L, n, torch.float64, 0)]
    P.run_many_device(seeds, n, n, *one)
    P.run_many_device(seeds, n, n, *two, None)
    torch.cuda.synchronize()
    for a, b in zip(one, two):
        assert torch.equal(a.all.view(torch.int64), b.all.view(torch.int64))
