"""Pair metrics at the sizes where their kernels and the staging change: the
batched FP64 call bit for bit against the oracle, the one-pair float call
against the oracle's restatement of the reference's arithmetic."""
import numpy as np
import pytest

import oracle as O
import svdb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,np_", [(1, 1), (63, 4), (64, 5), (65, 63), (130, 64), (257, 65),
                                   (128, 16_384), (33, 16_385), (20, 131_072), (3, 131_073),
                                   (2, (1 << 20) + 5)])
@pytest.mark.parametrize("deletes", [False, True])
def test_pair_batches(d, np_, deletes):
    """Row widths around a wavefront's 64 columns, pair counts around the four
    pairs of a turn, a block, a chunk and a staging block; a zero row (cosine
    NaN); deleted rows shift the indexes."""
    rng = np.random.default_rng(d + np_)
    X = rng.standard_normal((700, d))
    X[5] = 0.0
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    if deletes:
        for i in (3, 64, 600):
            db.delete(i)
            X = np.delete(X, i, axis=0)
    a = rng.integers(0, X.shape[0], np_)
    b = rng.integers(0, X.shape[0], np_)
    for m in ("l2", "cos", "dot"):
        got, want = db.pair_metrics(a, b, m), O.pairs_fp64(X, a, b, m)
        assert np.array_equal(np.isnan(got), np.isnan(want)), f"{d} {np_} {m}"
        ok = ~np.isnan(want)
        assert np.array_equal(got[ok].view(np.uint64), want[ok].view(np.uint64)), f"{d} {np_} {m}"
    # one bad index at the end: refused, and the next call is right again
    b[-1] = X.shape[0]
    with pytest.raises(Exception):
        db.pair_metrics(a, b, "dot")
    b[-1] = 0
    assert np.array_equal(db.pair_metrics(a, b, "dot"), O.pairs_fp64(X, a, b, "dot"))
    db.close()


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
