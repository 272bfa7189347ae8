"""PQ-flat searches ranked on the decoded rows (the fp16 GEMM, then the ADC of the codes it
admits) against the oracle's scan of every code: the path's row, depth and dimension edges,
odd code widths, filters, and the exact re-scan behind a failed certificate."""
import numpy as np
import pytest

import vdbg
from vdbg import datagen
from ivf_file import parse_pqflat

pytestmark = pytest.mark.gpu


def words(bits):
    w = np.zeros((len(bits) + 63) // 64 * 8, np.uint8)
    b = np.packbits(bits, bitorder="little")
    w[:b.size] = b
    return w.view(np.uint64)


# (batches of few rows score every code: test_ranked_few_rows has the batches that rank)
# rows at the path's limit of 1,024 and at remainders of the 64-row tiles; padded dims of one
# and several K chunks, with padding (100 -> 112, 20 -> 32) and without a kernel (400)
@pytest.mark.parametrize("n,dim,m,metric", [
    (1023, 64, 8, "l2"), (1024, 64, 8, "l2"), (1025, 100, 20, "cosine"), (4097, 20, 5, "l2"),
    (9000, 128, 16, "l2"), (9000, 128, 32, "ip"), (3001, 384, 48, "cosine"),
    (2000, 400, 16, "l2"), (70001, 96, 12, "l2")])
def test_ranked_search_matches_oracle(ctx, oracle, n, dim, m, metric):
    pd = vdbg.padded_dim(dim)
    base = datagen.clustered_unit(n, dim, 31, 32, 60, 0.6) * np.float32(3.0)
    q = datagen.pad(datagen.clustered_unit(131, dim, 33, 32, 60, 0.6) * np.float32(3.0), pd)
    rows = datagen.pad(base, pd)
    ds = vdbg.Dataset(ctx, rows, dim, metric)
    ix = vdbg.PqFlatIndex.build(ds, m, max_points=16, iters=2)
    pix = parse_pqflat(ix.save())
    rng = np.random.default_rng(7)
    ks = ctx.kernels
    # depths 0 (ADC order), up to the path's 240 and past it; 1, 33 and 131 queries
    for nq, k, rr, frac in ((1, 10, -1, None), (33, 10, -1, 0.4), (131, 24, 240, None),
                            (131, 10, 0, 0.01), (33, 24, 241, None), (33, 40, 0, None)):
        allow = None if frac is None else words(rng.random(n) < frac)
        print(f"n={n} dim={dim} m={m} {metric} nq={nq} k={k} rerank={rr} filter={frac}", flush=True)
        ids, d, dc = ix.search(q[:nq], k, rr, allow)
        od, oi, odc = oracle.pqflat_search(pix, rows, q[:nq], k, rr, metric, allow, kset=ks)
        assert np.array_equal(ids, oi)
        assert np.array_equal(d.view(np.uint32), od.view(np.uint32))
        assert np.array_equal(dc, odc)
    ix.close()
    ds.close()


# few rows rank only in batches large enough to repay it
@pytest.mark.parametrize("n,dim,m,metric", [(1024, 64, 8, "l2"), (1025, 100, 20, "cosine"),
                                            (4097, 20, 5, "l2")])
def test_ranked_few_rows(ctx, oracle, n, dim, m, metric):
    nq, k = 4500, 10
    print(f"ranked few rows n={n} dim={dim} m={m} {metric}", flush=True)
    pd = vdbg.padded_dim(dim)
    rows = datagen.pad(datagen.clustered_unit(n, dim, 31, 32, 60, 0.6) * np.float32(3.0), pd)
    q = datagen.pad(datagen.clustered_unit(nq, dim, 33, 32, 60, 0.6) * np.float32(3.0), pd)
    ds = vdbg.Dataset(ctx, rows, dim, metric)
    ix = vdbg.PqFlatIndex.build(ds, m, max_points=16, iters=2)
    at = np.r_[0:20, nq - 20:nq]
    for frac in (None, 0.4):
        allow = None if frac is None else words(np.random.default_rng(7).random(n) < frac)
        ids, d, dc = ix.search(q, k, 0, allow)
        assert ctx.last_gemm_bits() == 16
        od, oi, odc = oracle.pqflat_search(parse_pqflat(ix.save()), rows, q[at], k, 0, metric, allow,
                                           kset=ctx.kernels)
        assert np.array_equal(ids[at], oi) and np.array_equal(dc[at], odc)
        assert np.array_equal(d[at].view(np.uint32), od.view(np.uint32))
    ix.close()
    ds.close()


def test_duplicate_codes_and_fallbacks(ctx, oracle):
    """Rows sharing codes tie on the ADC (ids decide), a non-finite query has no certificate,
    and the forced exact re-scan returns the same results."""
    rows = datagen.sift_like(5000, 64, 41)
    rows[1000:3000] = rows[:2000]
    ds = vdbg.Dataset(ctx, rows, 64)
    ix = vdbg.PqFlatIndex.build(ds, 4, max_points=16, iters=2)
    pix = parse_pqflat(ix.save())
    q = datagen.sift_like(40, 64, 42)
    od, oi, odc = oracle.pqflat_search(pix, rows, q, 30, 120, "l2", None, kset=ctx.kernels)
    try:
        for level in (0, 1, 2):
            ctx.set_test_fallbacks(level)
            ids, d, dc = ix.search(q, 30, 120)
            assert np.array_equal(ids, oi), level
            assert np.array_equal(d.view(np.uint32), od.view(np.uint32)), level
            assert np.array_equal(dc, odc), level
        # every query re-scanned at the last level
        assert ctx.last_fallbacks() == 40
    finally:
        ctx.set_test_fallbacks(0)
    q[7, 3] = np.inf
    ids, d, _ = ix.search(q, 30, 120)
    keep = np.arange(40) != 7
    assert np.array_equal(ids[keep], oi[keep])
    ix.close()
    ds.close()


def test_decoded_rows_leave_memory_to_others(ctx):
    """An index whose decoded rows would take more than a quarter of the free memory goes without
    them: every code is scored, with the same answers."""
    import torch
    n, dim = 1200000, 128  # 312 MB of decoded rows
    print(f"decoded rows n={n}", flush=True)
    x = torch.randint(0, 200, (n, dim), generator=torch.Generator("cuda").manual_seed(3),
                      device="cuda").float()
    torch.cuda.synchronize()
    ds = vdbg.Dataset.from_device(ctx, x.data_ptr(), n, dim, dim)
    del x
    torch.cuda.empty_cache()
    q = np.random.default_rng(4).integers(0, 200, (40, dim)).astype(np.float32)
    want = None
    for left in (None, 1 << 30):
        fill = []
        while left is not None and torch.cuda.mem_get_info()[0] > left and len(fill) < 4:
            over = torch.cuda.mem_get_info()[0] - left  # (large allocations are rounded)
            try:
                fill.append(torch.empty(over, dtype=torch.uint8, device="cuda"))
            except torch.cuda.OutOfMemoryError:
                ds.close()
                pytest.skip("the free memory cannot be taken in one piece")
        ix = vdbg.PqFlatIndex.build(ds, 16, max_points=4, iters=1)
        del fill
        torch.cuda.empty_cache()
        ids, d, dc = ix.search(q, 10)
        assert ctx.last_gemm_bits() == (16 if left is None else 0)
        ix.close()
        if want is None:
            want = ids, d, dc
    assert np.array_equal(ids, want[0]) and np.array_equal(dc, want[2])
    assert np.array_equal(d.view(np.uint32), want[1].view(np.uint32))
    ds.close()


@pytest.mark.parametrize("n", [20000, 70001])
def test_routes_agree(ctx, oracle, n):
    """Calls on both sides of the choice between ranking and scoring every allowed code: few
    queries under a selective filter score (the filter's rows counted on the host, or on the
    device for a device call), the rest rank; the oracle's answers either way."""
    import torch
    rows, q = datagen.sift_like(n, 128, 51), datagen.sift_like(200, 128, 52)
    ds = vdbg.Dataset(ctx, rows, 128)
    ix = vdbg.PqFlatIndex.build(ds, 16, max_points=16, iters=2)
    pix = parse_pqflat(ix.save())
    rng = np.random.default_rng(8)
    seen = set()
    for nq, frac in ((1, 0.0), (1, 0.002), (7, 0.02), (33, 0.02), (200, 0.02), (200, 0.0625),
                     (1, 0.5), (33, None), (200, None)):
        print(f"routes n={n} nq={nq} filter={frac}", flush=True)
        allow = None if frac is None else words(rng.random(n) < frac)
        od, oi, odc = oracle.pqflat_search(pix, rows, q[:nq], 10, 100, "l2", allow,
                                           kset=ctx.kernels)
        ids, d, dc = ix.search(q[:nq], 10, 100, allow)
        bits = ctx.last_gemm_bits()
        seen.add(bits)
        assert np.array_equal(ids, oi) and np.array_equal(dc, odc)
        assert np.array_equal(d.view(np.uint32), od.view(np.uint32))
        dq = torch.from_numpy(q[:nq]).cuda()
        da = None if allow is None else torch.from_numpy(allow.view(np.int64)).cuda()
        di = torch.empty((nq, 10), dtype=torch.int32, device="cuda")
        dd = torch.empty((nq, 10), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        ix.search_device(dq.data_ptr(), nq, 10, 100, di.data_ptr(), dd.data_ptr(),
                         None if da is None else da.data_ptr())
        ctx.synchronize()
        assert ctx.last_gemm_bits() in (bits, 16)
        assert np.array_equal(di.cpu().numpy().view(np.uint32), oi)
        assert np.array_equal(dd.cpu().numpy().view(np.uint32), od.view(np.uint32))
    assert seen == {0, 16}
    ix.close()
    ds.close()
