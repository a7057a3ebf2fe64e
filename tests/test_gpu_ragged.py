"""Sampled runs whose rows start off the cache sectors against the same run in aligned rows, bit for bit.

Overlapping tiles store each row from its own first whole sector: every row alignment, base pointers
off the sectors, and sample counts at the edges of a tile, of a round and of its remainder.  What lies
between the rows' last sample and ld, and before the first row, stays as it was.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from mc_dagprop_amd import capi
from mc_dagprop_amd import workloads as wl

pytestmark = pytest.mark.gpu

ROUND = 256 * 120  # samples of one overlapping tile on each CU
FILL = 0xB3        # byte of memory that no result has been written to


class Rows:
    """A device array of rows with `first` elements before it, every byte FILL."""

    def __init__(self, rows: int, ld: int, dtype, first: int) -> None:
        self.dtype, self.shape, self.first = np.dtype(dtype), (rows, ld), first
        self.buf = capi.DeviceBuffer((first + rows * ld) * self.dtype.itemsize)
        capi.check(capi.lib().mcdp_memset(self.buf.ptr, FILL, self.buf.nbytes))
        self.ptr = ctypes.c_void_p(self.buf.ptr.value + first * self.dtype.itemsize)

    def bits(self) -> tuple[np.ndarray, np.ndarray]:
        """(the elements before the rows, the rows), as integers."""
        kind = np.uint64 if self.dtype.itemsize == 8 else np.uint32
        a = self.buf.to_array(kind, self.first + self.shape[0] * self.shape[1])
        return a[: self.first], a[self.first :].reshape(self.shape)


@pytest.fixture(scope="module")
def propagator():
    return capi.Propagator(wl.layered_vectorized(6, 100, 4, wl.network_dists(), 8, 77000))


def run(P, seeds: np.ndarray, ld: int, first: int, cause: bool = True) -> list[Rows]:
    out = [Rows(P.E, ld, np.float64, first), Rows(P.L, ld, np.float64, first)]
    if cause:
        out.append(Rows(P.E, ld, np.int32, first))
    d_seeds = capi.DeviceBuffer.from_array(seeds)
    P.run_many_device(d_seeds, len(seeds), ld, out[0], out[1], out[2] if cause else None)
    capi.check(capi.lib().mcdp_stream_synchronize(None))
    return out


@pytest.mark.parametrize(
    "n,pad,first",
    [(24_577, 0, 0), (27_005, 2, 1), (ROUND - 1, 0, 0), (ROUND, 3, 0), (ROUND + 1, 0, 3), (ROUND + 9, 4, 0),
     (32_767, 0, 0), (45_002, 1, 5), (2 * ROUND + 8, 5, 7), (2 * ROUND + 5003, 0, 2)],
)
def test_ragged_rows_equal_aligned_rows(gpu, propagator, n: int, pad: int, first: int) -> None:
    seeds = np.arange(n, dtype=np.int32) * 3 + 1
    want = run(propagator, seeds, (n + 15) // 16 * 16, 0)
    for got, ref in zip(run(propagator, seeds, n + pad, first), want):
        before, rows = got.bits()
        fill = np.frombuffer(bytes([FILL] * rows.dtype.itemsize), rows.dtype)[0]
        np.testing.assert_array_equal(rows[:, :n], ref.bits()[1][:, :n])
        assert (rows[:, n:] == fill).all() and (before == fill).all()


def test_without_causes(gpu, propagator) -> None:
    n = 33_001
    seeds = np.arange(n, dtype=np.int32)
    for a, b in zip(run(propagator, seeds, n, 0), run(propagator, seeds, n, 0, cause=False)):
        np.testing.assert_array_equal(a.bits()[1], b.bits()[1])
