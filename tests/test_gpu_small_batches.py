"""GPU parity of the low-precision search at the batch and row sizes where its
kernels change form: ids and FP64 scores equal the CPU FP64 oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
import svdb

pytestmark = pytest.mark.gpu


def check(db, X, Q, k, metric, precision):
    ids, sc = db.search(Q, k, metric, precision)
    rid, rsc = O.topk(X, Q, k, metric)
    what = f"{X.shape} {Q.shape[0]} queries k={k} {metric} {precision}"
    assert np.array_equal(ids, rid), f"{what}: ids differ"
    assert np.array_equal(sc.view(np.uint64), rsc.view(np.uint64)), f"{what}: scores differ"


@pytest.mark.parametrize("precision,d", [("bf16", 1), ("bf16", 2), ("bf16", 15), ("bf16", 17),
                                         ("bf16", 33), ("bf16", 255), ("bf16", 257),
                                         ("bf16", 1536), ("fp8", 3), ("fp8", 255), ("fp8", 257),
                                         ("fp8", 1533)])
def test_query_prep_widths(precision, d):
    """Query widths either side of the prep kernel's 16-column chain steps and
    256-column loads, odd ones among them; 1, 4 and 5 queries (its blocks
    hold 4) and a zero query."""
    rng = np.random.default_rng(d)
    X = rng.standard_normal((3000, d))
    Q = rng.standard_normal((5, d))
    Q[2] = 0.0
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    if precision == "fp8":
        db.enable_shadow("fp8")
    for nq in (1, 4, 5):
        for metric in ("l2", "cos", "dot"):
            check(db, X, Q[:nq], 7, metric, precision)
    db.close()
