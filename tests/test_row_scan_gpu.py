"""Batches of at most 8 queries over rows of any values (k_row_scan and its merge; from 3 queries
on only rows without a GEMM kernel take it) against the oracle: the tile and chunk edges, padded dims with and without a GEMM kernel, filters, ties,
queries without a bound, and the exact re-scan behind the certificate."""
import numpy as np
import pytest

import vdbg
from vdbg import datagen

pytestmark = pytest.mark.gpu


def words(bits):
    w = np.zeros((len(bits) + 63) // 64 * 8, np.uint8)
    b = np.packbits(bits, bitorder="little")
    w[:b.size] = b
    return w.view(np.uint64)


def check(got, want):
    assert np.array_equal(got[0], want[1])
    assert np.array_equal(got[1].view(np.uint32), want[0].view(np.uint32))


# rows around a mask word, the 1,024-row tile and several chunks; dims of one partial, one and
# several 64-dim runs (16, 48, 100 -> 112, 384), past the fp16 unroll (512, 848) and integers
# at a width the int8 kernels do not take; 1 to 8 queries; k up to 48
@pytest.mark.parametrize("n,dim,nq,k,metric,data", [
    (1, 16, 1, 1, "l2", "uniform"), (291, 839, 1, 10, "cosine", "unit"),
    (1000, 64, 1, 7, "ip", "uniform"), (999, 64, 1, 7, "l2", "uniform"), (63, 48, 3, 10, "ip", "uniform"),
    (65, 100, 8, 48, "cosine", "unit"), (1023, 384, 2, 10, "cosine", "unit"),
    (1025, 384, 1, 48, "cosine", "unit"), (20001, 100, 5, 10, "cosine", "unit"),
    (70003, 128, 4, 20, "l2", "uniform"), (30000, 512, 1, 1, "l2", "uniform"),
    (9001, 839, 2, 13, "cosine", "unit"), (9001, 839, 3, 13, "l2", "sift"),
    (40000, 96, 8, 10, "l2", "sift"), (300000, 16, 7, 10, "ip", "uniform")])
def test_row_scan(ctx, oracle, n, dim, nq, k, metric, data):
    print(f"row scan n={n} dim={dim} nq={nq} k={k} {metric} {data}", flush=True)
    pd = vdbg.padded_dim(dim)
    if data == "sift":
        base, qs = datagen.sift_like(n, dim, 161), datagen.sift_like(nq, dim, 162)
    elif data == "uniform":
        base, qs = datagen.uniform_rows(n, dim, 163), datagen.uniform_rows(nq, dim, 164)
    else:
        base = datagen.clustered_unit(n, dim, 165, 166, 80, 0.7)
        qs = datagen.clustered_unit(nq, dim, 167, 166, 80, 0.7)
    base, qs = datagen.pad(base, pd), datagen.pad(qs, pd)
    ds = vdbg.Dataset(ctx, base, dim, metric)
    rng = np.random.default_rng(n)
    # no filter, most rows, few, (almost) none
    for frac in (None, 0.97, 0.03, 2.0 / n):
        allow = None if frac is None else words(rng.random(n) < frac)
        want = oracle.flat_search(base, qs, k, metric=metric, allow=allow)
        check(ds.flat_search(qs, k, allow=allow), want)
        try:
            ctx.set_test_fallbacks(2)
            check(ds.flat_search(qs, k, allow=allow), want)
            few = n < 1024 and n * (256 + pd) < 320000 + 80000 * (nq - 1)  # scored exactly
            assert ctx.last_fallbacks() == nq or allow is not None or few
            ctx.set_gated_fallbacks(False)
            check(ds.flat_search(qs, k, allow=allow), want)
        finally:
            ctx.set_test_fallbacks(0)
            ctx.set_gated_fallbacks(True)
    try:  # from the fp32 rows
        ctx.set_fp16_gemm(False)
        check(ds.flat_search(qs, k), oracle.flat_search(base, qs, k, metric=metric))
    finally:
        ctx.set_fp16_gemm(True)
    ds.close()


def test_row_scan_ties_and_queries_without_a_bound(ctx, oracle):
    """Rows repeated 40 times tie on the distance (the smaller row wins, past what a chunk
    keeps); a query of huge values overflows its keys and bound, one with a NaN has none."""
    base = np.repeat(datagen.uniform_rows(500, 48, 171), 40, axis=0)
    qs = datagen.uniform_rows(6, 48, 172)
    qs[1] *= np.float32(1e30)
    ds = vdbg.Dataset(ctx, base, 48)
    check(ds.flat_search(qs, 45), oracle.flat_search(base, qs, 45))
    qs[2, 5] = np.nan
    ids, d = ds.flat_search(qs, 10)
    od, oi = oracle.flat_search(base, qs, 10)
    keep = [0, 1, 3, 4, 5]
    check((ids[keep], d[keep]), (od[keep], oi[keep]))
    ds.close()


def test_row_scan_appendable(ctx, oracle):
    """Appended rows (no fp16 copy) from the first row on."""
    ds = vdbg.Dataset.appendable(ctx, 40, "l2", capacity=64)
    base = datagen.pad(datagen.uniform_rows(3000, 40, 181), 48)
    qs = datagen.pad(datagen.uniform_rows(3, 40, 182), 48)
    at = 0
    for step in (1, 7, 56, 1, 935, 2000):
        ds.append(base[at:at + step])
        at += step
        check(ds.flat_search(qs, 12), oracle.flat_search(base[:at], qs, 12))
    ds.close()
