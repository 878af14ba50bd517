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


@pytest.mark.parametrize("n,d,nq,k,short", [
    (1, 5, 3, 4, None),       # fewer rows than k
    (40, 64, 2, 40, None),    # k is every row
    (700, 65, 1, 1, 256),     # a shortlist far wider than k: the second round
    (700, 63, 5, 128, 256),
    (900, 16, 4, 17, 17),     # the shortlist is k
    (900, 129, 1030, 10, 64), # a bulk batch: k rows, then what their k-th leaves
    (900, 8, 1024, 128, None),
])
def test_rerank_shapes(n, d, nq, k, short):
    """Row counts, widths, k and shortlist widths around the first-stage
    rerank's rounds (16 rows, 64 columns, 1,024 queries), over a store with
    duplicated rows (ties by id) and with degenerate rows, which enter every
    query's candidates, also when they are its answer."""
    rng = np.random.default_rng(n + d)
    X = rng.integers(-3, 4, size=(n, d)).astype(np.float64)
    if n > 4:
        X[n // 2:] = X[:n - n // 2]
        X[1] = 0.0
        X[n - 1] = 0.0
        X[2] = 1e30
    Q = rng.integers(-3, 4, size=(nq, d)) + 0.125 * rng.standard_normal((nq, d))
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    if short:
        db.set_shortlist(short)
    for metric in ("l2", "cos", "dot"):
        check(db, X, Q, k, metric, "bf16")
    db.close()


@pytest.mark.parametrize("d,nq", [(30, 70), (64, 5), (128, 600), (129, 130), (256, 300),
                                  (500, 40), (768, 130), (1536, 70)])
def test_thresholded_lists(d, nq):
    """Row and query counts over which the first pass starts from a sample's
    threshold, every padded width, ragged last tile; k on both sides of the
    wider shortlist.  A third of the rows are one cluster stored in a row, so
    that the lists of the slices it lies in fill up."""
    rng = np.random.default_rng(d)
    n = 20_011
    X = rng.standard_normal((n, d))
    X[5000:5000 + n // 3] = X[0] + 0.05 * rng.standard_normal((n // 3, d))
    Q = np.vstack([X[0] + 0.05 * rng.standard_normal((nq // 2, d)),
                   rng.standard_normal((nq - nq // 2, d))])
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    for metric in ("l2", "cos", "dot"):
        for k in (10, 40):
            check(db, X, Q, k, metric, "bf16")
    if d <= 256:
        ids, sc = db.search(Q, 10, [("l2", "cos", "dot")[i % 3] for i in range(nq)], "bf16")
        for j, metric in enumerate(("l2", "cos", "dot")):
            rid, rsc = O.topk(X, Q[j::3], 10, metric)
            assert np.array_equal(ids[j::3], rid) and np.array_equal(sc[j::3], rsc), metric
    if d >= 500:
        db.enable_shadow("fp8")
        for metric in ("l2", "cos", "dot"):
            check(db, X, Q, 10, metric, "fp8")
    db.close()


@pytest.mark.parametrize("d,nq,k", [(20, 11_777, 2), (256, 5_800, 10)])
def test_slices_past_two_rounds(d, nq, k):
    """Query counts whose blocks leave a last round of the GPU part empty at
    the fewest slices, so that the scan takes more of them; ids and scores as
    the exhaustive FP64 search has them.  A third of the rows are one cluster
    stored in a row."""
    rng = np.random.default_rng(d)
    n = 100_003
    X = rng.standard_normal((n, d))
    X[5000:5000 + n // 3] = X[0] + 0.05 * rng.standard_normal((n // 3, d))
    Q = np.vstack([X[0] + 0.05 * rng.standard_normal((nq // 8, d)),
                   rng.standard_normal((nq - nq // 8, d))])
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    for metric in ("l2", "cos", "dot"):
        ids, sc = db.search(Q, k, metric, "bf16")
        rid, rsc = db.search(Q, k, metric, "fp64")
        assert np.array_equal(ids, rid), f"{d} {nq} {metric}: ids differ"
        assert np.array_equal(sc.view(np.uint64), rsc.view(np.uint64)), f"{d} {nq} {metric}"
    db.close()


@pytest.mark.parametrize("d", [30, 64, 128, 200])
def test_query_counts_at_the_fragments_edges(d):
    """Query counts at which the first-pass scan changes the queries of a block
    and of a wavefront, single-metric and mixed."""
    rng = np.random.default_rng(d)
    n = 20_011
    X = rng.standard_normal((n, d))
    X[7000:7000 + n // 4] = X[0] + 0.1 * rng.standard_normal((n // 4, d))
    Q = np.vstack([X[0] + 0.1 * rng.standard_normal((100, d)), rng.standard_normal((157, d))])
    Q = Q[rng.permutation(257)]
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    want = {m: O.topk(X, Q, 10, m) for m in ("l2", "cos", "dot")}
    for nq in (16, 17, 128, 129, 256, 257):
        for m in ("l2", "cos", "dot"):
            ids, sc = db.search(Q[:nq], 10, m, "bf16")
            assert np.array_equal(ids, want[m][0][:nq]), f"{d} {nq} {m}"
            assert np.array_equal(sc, want[m][1][:nq]), f"{d} {nq} {m}"
        ms = [("l2", "cos", "dot")[i % 3] for i in range(nq)]
        ids, sc = db.search(Q[:nq], 10, ms, "bf16")
        for i, m in enumerate(ms):
            assert np.array_equal(ids[i], want[m][0][i]) and np.array_equal(sc[i], want[m][1][i]), f"{d} {nq} mixed {i}"
    db.close()


@pytest.mark.parametrize("nq", [40, 3000])
def test_candidate_lists_within_a_budget(nq):
    """A device-memory budget that leaves no room for the scan's usual lists:
    fewer slices, the same answers; without any room the search is refused,
    and answered again once the budget is lifted."""
    rng = np.random.default_rng(nq)
    X = rng.standard_normal((40_007, 64))
    Q = rng.standard_normal((nq, 64))
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    want = O.topk(X, Q, 10, "l2")
    lists = nq * 8 * 4 * 17 * 8  # 8 slices' lists
    rest = nq * (64 * 8 + 64 * 2 + 64 * 8 + 10 * 12 + 256) + (2 << 20)
    db.set_budget(db.stats()["device_bytes"] + lists + rest)
    ids, sc = db.search(Q, 10, "l2", "bf16")
    assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])
    db.close()
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    db.set_budget(db.stats()["device_bytes"] + 4096)
    with pytest.raises(Exception):
        db.search(Q, 10, "l2", "bf16")
    db.set_budget(0)
    ids, sc = db.search(Q, 10, "l2", "bf16")
    assert np.array_equal(ids, want[0]) and np.array_equal(sc, want[1])
    db.close()


def pages(*sizes):
    return sum((max(int(b), 1) + 4095) // 4096 * 4096 for b in sizes)


def first_pass_scratch(nq, k, dp, qpb, lists, L):
    """Device scratch of a first pass whose lists hold 8 entries of 8 bytes, for
    queries and results in device memory."""
    pad = (nq + qpb - 1) // qpb * qpb
    return pages((pad + qpb) * dp * 2, pad * 48, lists * 32, lists * 32, nq * L * 4, nq * L * 4,
                 nq * 4, (nq + 3) * 4, nq * 8, nq * k * 8, nq * k * 4, nq * 4, nq * 4)


@pytest.mark.parametrize("n,d,nq,k", [(4000, 64, 3000, 5), (4000, 250, 2000, 1),
                                      (30_000, 60, 700, 10), (30_000, 128, 400, 100)])
def test_lists_of_eight_entries_fit(n, d, nq, k):
    """A device-memory budget that holds 8 slices' lists of eight entries, with
    nothing besides, on stores with and without a sample's threshold."""
    rng = np.random.default_rng(n + nq)
    X = rng.standard_normal((n, d))
    Q = rng.standard_normal((nq, d))
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    dQ = svdb.DeviceArray.from_host(Q)
    ids = svdb.DeviceArray((nq, k), np.uint64)
    sc = svdb.DeviceArray((nq, k), np.float64)
    dp = 64 if d <= 64 else 128 if d <= 128 else 256
    L = 64 if k <= 32 else 256
    lists = nq * 4 * (128 if k > 32 else 8)
    db.set_budget(db.stats()["device_bytes"] +
                  first_pass_scratch(nq, k, dp, 512 if dp < 256 else 256, lists, L))
    error = svdb.lib().svdb_last_error()
    db.search_device(dQ.ptr, nq, d, k, "dot", "bf16", ids.ptr, sc.ptr)
    rid, rsc = O.topk(X, Q, k, "dot")
    assert np.array_equal(ids.to_host(), rid) and np.array_equal(sc.to_host(), rsc)
    assert svdb.lib().svdb_last_error() == error  # the smaller plan's is no error
    for a in (dQ, ids, sc):
        a.free()
    db.close()


@pytest.mark.parametrize("n,nq", [(4000, 300), (40_007, 300), (40_007, 3000)])
def test_fallback_within_a_budget(n, nq):
    """A zero query, which only the FP64 scan can answer, in a batch under a budget
    that holds lists of eight entries, the retries' buffers and that scan's: the
    lists must not take what those need."""
    rng = np.random.default_rng(n + nq)
    d, k = 64, 10
    X = rng.standard_normal((n, d))
    Q = rng.standard_normal((nq, d))
    Q[nq // 2] = 0.0
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    tiles = (n + 127) // 128
    slices = min(512 // ((nq + 511) // 512) // 8 * 8, max(8, (tiles // 4 + 7) // 8 * 8))
    retries = pages(1024 * 4, 1024 * 4, 4, 16, 4096 * 4, 4096 * 4)
    exact = pages(d * 8, k * 8, k * 8, 4, 4 * max(8, n // 1024) * k * 8, 4 * max(8, n // 1024) * k * 4, 24)
    db.set_budget(db.stats()["device_bytes"] + pages(nq * d * 8, nq * k * 8, nq * k * 8) +
                  first_pass_scratch(nq, k, 64, 512, nq * 4 * slices, 64) + retries + exact)
    error = svdb.lib().svdb_last_error()
    for metric in ("l2", "dot"):
        check(db, X, Q, k, metric, "bf16")
        assert db.stats()["fallbacks"] > 0
        assert svdb.lib().svdb_last_error() == error  # the smaller plan's is no error
    db.close()


def test_lists_make_room_for_rows():
    """What searches leave behind in device memory does not stand in the way of
    rows or of another kind of search."""
    rng = np.random.default_rng(5)
    X = rng.standard_normal((20_000, 32))
    Q = rng.standard_normal((4000, 32))
    db = svdb.Database(kd_dimension=1)
    db.bulk_insert(X)
    db.search(Q, 10, "l2", "bf16")
    db.search(Q, 10, "l2", "fp64")
    db.set_budget(db.stats()["device_bytes"] + (1 << 20))
    db.bulk_insert(rng.standard_normal((15_000, 32)))  # the store doubles
    db.set_budget(0)
    ids, sc = db.search(Q[:50], 10, "l2", "bf16")
    rid, rsc = db.search(Q[:50], 10, "l2", "fp64")
    assert np.array_equal(ids, rid) and np.array_equal(sc, rsc)
    db.close()
