"""Answers deeper than 240: the ranking GEMM's candidates scored and sorted by one block per
query, the block sort of every row's key for small segments, and the scan of every row behind a
failed certificate, against the oracle."""
import numpy as np
import pytest

import vdbg
from vdbg import datagen

pytestmark = pytest.mark.gpu


def check(gi, gd, oi, od):
    assert np.array_equal(gi, oi)
    assert np.array_equal(gd.view(np.uint32), od.view(np.uint32))


def words(bits):
    w = np.zeros((len(bits) + 63) // 64 * 8, np.uint8)
    b = np.packbits(bits, bitorder="little")
    w[:b.size] = b
    return w.view(np.uint64)


# the block sort's limit of 16,384 rows, its padding to powers of two, and the ranked path's
# depths from 241 to where its sample is too small for them (10,000 of 30,000 rows)
@pytest.mark.parametrize("n,dim,nq,k,metric,data,frac", [
    (129, 32, 3, 241, "l2", "sift", None), (4096, 32, 5, 4096, "l2", "sift", None),
    (16384, 20, 33, 1000, "ip", "uniform", 0.7), (16385, 20, 33, 241, "ip", "uniform", 0.7),
    (20001, 100, 61, 1000, "cosine", "unit", 0.98), (70001, 128, 130, 1000, "l2", "sift", None),
    (70001, 128, 7, 300, "l2", "sift", 0.6), (118385, 100, 61, 3000, "cosine", "unit", None),
    (30000, 48, 5, 10000, "l2", "uniform", None), (40000, 400, 3, 700, "l2", "uniform", None)])
def test_deep_flat(ctx, oracle, n, dim, nq, k, metric, data, frac):
    print(f"deep flat n={n} dim={dim} nq={nq} k={k} {metric} {data} filter={frac}", flush=True)
    pd = vdbg.padded_dim(dim)
    if data == "sift":
        base, qs = datagen.sift_like(n, dim, 61), datagen.sift_like(nq, dim, 62)
    elif data == "uniform":
        base, qs = datagen.uniform_rows(n, dim, 63), datagen.uniform_rows(nq, dim, 64)
    else:
        base = datagen.clustered_unit(n, dim, 65, 66, 80, 0.7)
        qs = datagen.clustered_unit(nq, dim, 67, 66, 80, 0.7)
    base, qs = datagen.pad(base, pd), datagen.pad(qs, pd)
    allow = None if frac is None else words(np.random.default_rng(3).random(n) < frac)
    ds = vdbg.Dataset(ctx, base, dim, metric)
    od, oi = oracle.flat_search(base, qs, k, metric=metric, allow=allow)
    check(*ds.flat_search(qs, k, allow=allow), oi, od)
    try:  # every answer re-scanned: the same results
        ctx.set_test_fallbacks(1)
        check(*ds.flat_search(qs[:3], k, allow=allow), oi[:3], od[:3])
    finally:
        ctx.set_test_fallbacks(0)
    ds.close()


def test_deep_batch_in_parts(ctx, oracle):
    """More queries than one pass's scratch is planned for (some 1,300 at 16,384 keys a query)."""
    n, dim, nq, k = 70000, 16, 2050, 5000
    base, qs = datagen.uniform_rows(n, dim, 71), datagen.uniform_rows(nq, dim, 72)
    ds = vdbg.Dataset(ctx, base, dim)
    gi, gd = ds.flat_search(qs, k)
    at = np.r_[0:4, 2040:2050]
    od, oi = oracle.flat_search(base, qs[at], k)
    check(gi[at], gd[at], oi, od)
    ds.close()


def test_deep_sample_short_of_depth(ctx, oracle):
    """Every near row on a sampled position: the threshold keeps fewer rows than the depth, the
    certificate refuses and every row is scored."""
    n, dim, near = 4 * 65536, 32, 600
    rng = np.random.default_rng(81)
    base = (100.0 + rng.random((n, dim), dtype=np.float32)).astype(np.float32)
    at = (n // 2048) * np.arange(near)
    base[at, :] = 0.0
    base[at, 0] = 0.01 * (1 + np.arange(near, dtype=np.float32))
    qs = np.zeros((5, dim), np.float32)
    qs[:, 1] = 1e-3 * np.arange(5, dtype=np.float32)
    ds = vdbg.Dataset(ctx, base, dim)
    gi, gd = ds.flat_search(qs, 1000)
    od, oi = oracle.flat_search(base, qs, 1000)
    assert ctx.last_fallbacks() > 0
    check(gi, gd, oi, od)
    ds.close()


@pytest.mark.parametrize("n,depth", [(16000, 700), (50000, 241), (50000, 2000)])
def test_deep_sq8(ctx, oracle, n, depth):
    base, qs = datagen.uniform_rows(n, 112, 91), datagen.uniform_rows(37, 112, 92)
    print(f"deep sq8 n={n} depth={depth}", flush=True)
    ds = vdbg.Dataset(ctx, base, 112)
    sq = vdbg.Sq8Index(ds)
    od, oi = oracle.sq8_search(base, sq.codes(), sq.vmin, sq.scale, qs, 10, depth)
    check(*sq.search(qs, 10, depth), oi, od)
    sq.close()
    ds.close()


# A deep answer's rows lie together.  61 queries: the candidates' segments hold every row of
# their half chunks, so no answer is re-scanned; 900: the segments are sized for rows in any order,
# and the queries that overflow them are scored over every row in one batch.
@pytest.mark.parametrize("nq", [61, 900])
@pytest.mark.parametrize("kind", ["flat", "sq8"])
def test_deep_rows_stored_by_cluster(ctx, oracle, nq, kind):
    n, dim, k, per = 118385, 112, 1000, 1500
    print(f"deep, rows by cluster, {kind} nq={nq}", flush=True)
    rng = np.random.default_rng(95)
    centers = rng.random((n // per + 1, dim), dtype=np.float32)
    base = np.repeat(centers, per, axis=0)[:n]
    base += 0.2 * rng.standard_normal((n, dim), dtype=np.float32)
    qs = centers[rng.integers(0, n // per, nq)]
    qs = (qs + 0.2 * rng.standard_normal((nq, dim), dtype=np.float32)).astype(np.float32)
    qs[: nq // 2] = rng.random((nq // 2, dim), dtype=np.float32)  # (no cluster of their own)
    at = np.r_[0:8, nq - 8 : nq]
    ds = vdbg.Dataset(ctx, base, dim)
    if kind == "flat":
        gi, gd = ds.flat_search(qs, k)
        again = ctx.last_fallbacks()
        od, oi = oracle.flat_search(base, qs[at], k)
    else:
        sq = vdbg.Sq8Index(ds)
        gi, gd = sq.search(qs, 10, k)
        again = ctx.last_fallbacks()
        od, oi = oracle.sq8_search(base, sq.codes(), sq.vmin, sq.scale, qs[at], 10, k)
        sq.close()
    check(gi[at], gd[at], oi, od)
    assert again == 0 if nq == 61 else 0 < again < nq
    ds.close()
