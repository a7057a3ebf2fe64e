"""Quantiles by value bins: every way a rank's bin is resolved, bit for bit against the statistics oracle.

* few small bins: the open ranks' bins gathered together (at most 512 keys in at most 8 bins);
* one bin after another: too many bins or keys for that, bins of one value and of several;
* bins with more keys than are gathered: of one value (settled by their extremes), of two signed
  zeros or of neighbouring values (left to the radix passes).
"""

from __future__ import annotations

import numpy as np
import pytest

import dags as D
import oracle
from mc_dagprop_amd import capi
from test_gpu_stats import assert_quantiles_equal, bits, run_stats_device

pytestmark = pytest.mark.gpu


def rows(rng: np.random.Generator, n: int) -> np.ndarray:
    centre = rng.normal(0.0, 1.0, n)
    mass = (n - 2) * 2 // 3
    wide = np.array([-1000.0, 1000.0])  # sets the width of a bin, about 0.49

    def around(middle: np.ndarray) -> np.ndarray:
        return np.concatenate([wide, middle, rng.uniform(-1000.0, 1000.0, n - 2 - len(middle))])

    cols = [
        centre,
        np.exp(centre),
        np.round(centre, 1),
        np.round(centre, 2),
        around(np.full(mass, 0.25)),
        around(rng.choice([0.25, 0.3], mass)),
        around(rng.choice([0.25, np.nextafter(0.25, 1.0)], mass)),
        around(rng.choice([-0.0, 0.0], mass)),
        around(rng.uniform(0.25, 0.45, mass)),
        np.sort(rng.uniform(-1.0, 1.0, n)),
        np.where(rng.random(n) < 0.5, -7.0, np.where(rng.random(n) < 0.5, 3.0, rng.uniform(-7.0, 3.0, n))),
    ]
    return np.stack([c if i == 9 else rng.permutation(c) for i, c in enumerate(cols)], axis=1)


@pytest.mark.parametrize(
    "q",
    [[0.5], [0.25, 0.5, 0.99], [0.01, 0.2, 0.4, 0.45, 0.55, 0.6, 0.8, 0.999]],
    ids=["one", "three", "eight"],
)
@pytest.mark.parametrize("n", [3, 64, 511, 513, 1000, 2049, 4095, 16_000, 70_001])
def test_quantiles_by_value_bins(gpu, n: int, q: list[float]) -> None:
    rng = np.random.default_rng(n)
    r = rows(rng, n)
    dag = D.parity_long_chain(r.shape[1] - 1)
    P = capi.Propagator(dag)
    assert P.E == r.shape[1]
    c = np.full(r.shape, -1, dtype=np.int32)
    mean, quant, _ = run_stats_device(P, r, c, q, pad=3)
    om, oq, _ = oracle.event_stats(r, c, oracle.pred_sources(dag), q)
    assert_quantiles_equal(quant, oq)
    np.testing.assert_array_equal(bits(mean), bits(om))
