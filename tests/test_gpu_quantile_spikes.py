"""Quantiles of rows with a value held by many samples among close others, in value bins of more keys than are
gathered: ranks below, in and above that value's mass, bit for bit against the statistics oracle."""

from __future__ import annotations

import numpy as np
import pytest

import dags as D
import oracle
from mc_dagprop_amd import capi
from test_gpu_stats import assert_quantiles_equal, run_stats_device

pytestmark = pytest.mark.gpu

SHARES = [(0.1, 0.5, 0.1), (0.0, 0.6, 0.05), (0.05, 0.6, 0.0), (0.3, 0.2, 0.3), (0.45, 0.02, 0.45), (0.0, 0.9, 0.0)]


def spiked(rng: np.random.Generator, n: int, below: float, mass: float, above: float, value: float) -> np.ndarray:
    """Shares of samples just below, at and just above `value`, all in one bin; the rest spread over [-1000, 1000]."""
    parts = [np.array([-1000.0, 1000.0]), np.full(int(n * mass), value),
             value - rng.uniform(1e-9, 1e-3, int(n * below)), value + rng.uniform(1e-9, 1e-3, int(n * above))]
    used = sum(map(len, parts))
    return rng.permutation(np.concatenate(parts + [rng.uniform(-1000.0, 1000.0, max(0, n - used))])[:n])


@pytest.mark.parametrize("n", [4096, 5003, 30_011, 131_073])
def test_ranks_around_a_spike(gpu, n: int) -> None:
    rng = np.random.default_rng(n)
    rows = [spiked(rng, n, *s, value) for s in SHARES for value in (0.25, -0.0)]
    # two such values in one bin, and two in different bins
    rows += [rng.permutation(np.concatenate([spiked(rng, n // 2, 0.1, 0.6, 0.1, 0.2), spiked(rng, n - n // 2, 0.1, 0.6, 0.1, v)]))
             for v in (0.3, 400.0)]
    rows.append(np.sort(rows[0]))
    r = np.stack(rows, axis=1)
    middle = [float(np.mean(r[:, 0] < 0.25)), float(np.mean(r[:, 0] <= 0.25))]  # edges of the first row's mass
    dag = D.parity_long_chain(r.shape[1] - 1)
    P = capi.Propagator(dag)
    c = np.full(r.shape, -1, dtype=np.int32)
    for q in ([0.5], [0.05, 0.3, 0.5, 0.62, 0.7, 0.9], middle + [middle[0] + 1e-4, middle[1] - 1e-4]):
        _, quant, _ = run_stats_device(P, r, c, q, pad=1)
        _, want, _ = oracle.event_stats(r, c, oracle.pred_sources(dag), q)
        assert_quantiles_equal(quant, want)
