"""Pair metrics at the sizes where their kernels and the staging change: the
batched FP64 call bit for bit against the oracle, the one-pair float call
against the oracle's restatement of the reference's arithmetic."""
import numpy as np
import pytest

import oracle as O
import svdb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 8, 9, 63, 64, 65, 255, 256, 257, 264, 511, 1536])
def test_float_metrics_widths(n):
    """Lengths around the 64 lanes that take the products, the chains' steps of
    eight and the 256 columns held at a time."""
    rng = np.random.default_rng(n)
    A = rng.standard_normal((12, n)) * rng.choice([1e-3, 1.0, 1e3], (12, 1))
    A[2, n - 1] = np.inf
    A[3] = 0.0
    ia, ib = np.arange(0, 12, 2, dtype=np.uint64), np.arange(1, 12, 2, dtype=np.uint64)
    for metric in ("cos", "l2", "dot"):
        want = O.ref_pairs(A, ia, ib, metric).astype(np.float32)
        got = np.array([svdb.legacy_metric(A[i], A[j], metric) for i, j in zip(ia, ib)],
                       dtype=np.float32)
        assert np.array_equal(np.isnan(got), np.isnan(want)), f"{n} {metric}"
        ok = ~np.isnan(want)
        assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32)), f"{n} {metric}"
