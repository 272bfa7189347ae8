"""Collection searches of at most 8 queries over flat segments (every segment scored in one
launch under its mask) against the oracle's composition of the per-segment searches: segments
of one row to several chunks, empty ones and empty filters, ids held by two segments, the
largest number of segments and one more, and the re-scan of the segments behind uncertified
answers."""
import numpy as np
import pytest

import vdbg
from vdbg import datagen

pytestmark = pytest.mark.gpu


def mask(n, frac, seed):
    bits = np.random.default_rng(seed).random(n) < frac
    w = np.zeros((n + 63) // 64 * 8, np.uint8)
    b = np.packbits(bits, bitorder="little")
    w[:b.size] = b
    return w.view(np.uint64)


def build(ctx, sizes, dim, metric, data, seed):
    pd = vdbg.padded_dim(dim)
    segs, handles, nxt = [], [], 10
    for i, n in enumerate(sizes):
        if data == "sift":
            x = datagen.sift_like(n, dim, seed + i)
        else:
            x = datagen.clustered_unit(n, dim, seed + i, 79, 40, 0.5)
        base = datagen.pad(x, pd)
        ext = np.arange(nxt, nxt + n, dtype=np.uint64) * 7
        nxt += n
        if i == 2 and n >= 50:
            ext[:50] = segs[0]["ext"][:50]  # an upsert visible in both segments
            base[:50] = segs[0]["base"][:50]
        ds = vdbg.Dataset(ctx, base, dim, metric)
        if n:
            ds.set_external_ids(ext)
        segs.append({"base": base, "ext": ext, "kind": "flat", "deleted": None, "filter": None})
        handles.append(ds)
    return segs, handles


def run(ctx, oracle, segs, handles, dim, metric, raw, k):
    got = vdbg.collection_search(
        ctx, [(ds, None, sg["deleted"], sg["filter"]) for ds, sg in zip(handles, segs)], dim,
        metric, raw, k)
    want = oracle.collection_search(segs, dim, metric, raw, k)
    assert got[3] == want[3]
    assert np.array_equal(got[0], want[0])
    assert np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32))
    assert np.array_equal(got[2], want[2])


@pytest.mark.parametrize("sizes,dim,metric,data", [
    ([5000, 1, 3000, 64, 1025, 30000], 96, "cosine", "unit"),
    ([2000, 700, 900], 100, "l2", "unit"), ([4000, 50000], 128, "l2", "sift"),
    ([3000], 384, "cosine", "unit"), ([100] * 16, 48, "ip", "unit"),
    ([100] * 17, 48, "ip", "unit")])
def test_small_collection(ctx, oracle, sizes, dim, metric, data):
    segs, handles = build(ctx, sizes, dim, metric, data, 300)
    rng = np.random.default_rng(5)
    for nq, k, filt, deleted in ((1, 10, None, None), (1, 10, 0.1, 0.02), (2, 48, 0.5, None),
                                 (3, 1, 0.05, 0.3), (8, 10, None, 0.02), (8, 49, 0.2, None)):
        print(f"small collection {sizes} nq={nq} k={k} filter={filt} deleted={deleted}", flush=True)
        for i, sg in enumerate(segs):
            n = sizes[i]
            sg["filter"] = None if filt is None else mask(n, filt if i != 1 else 0.0, 20 + i)
            sg["deleted"] = None if deleted is None else mask(n, deleted, 40 + i)
        if data == "sift":
            raw = datagen.sift_like(nq, dim, int(rng.integers(1000)))
        else:
            raw = datagen.clustered_unit(nq, dim, int(rng.integers(1000)), 79, 40, 0.5) * 3
            raw = raw.astype(np.float32)
        run(ctx, oracle, segs, handles, dim, metric, raw, k)
        try:  # no answer certified: every segment re-scanned
            ctx.set_test_fallbacks(1)
            run(ctx, oracle, segs, handles, dim, metric, raw, k)
        finally:
            ctx.set_test_fallbacks(0)
    bad = raw.copy()
    bad[0, 3] = np.inf
    with pytest.raises(vdbg.VdbgError) as e:
        run(ctx, oracle, segs, handles, dim, metric, bad, 10)
    assert e.value.code == 1 and "NaN or infinite" in str(e.value)
    for ds in handles:
        ds.close()


def test_small_collection_device_results(ctx, oracle):
    """Queries and results in device memory, on a stream of the caller's."""
    import torch
    segs, handles = build(ctx, [4000, 2500, 9000], 96, "cosine", "unit", 500)
    for i, sg in enumerate(segs):
        sg["filter"] = mask(sg["base"].shape[0], 0.2, 60 + i)
    raw = (datagen.clustered_unit(2, 96, 71, 79, 40, 0.5) * 3).astype(np.float32)
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        q = torch.from_numpy(raw).cuda()
        ids = torch.empty((2, 10), dtype=torch.int64, device="cuda")
        d = torch.empty((2, 10), dtype=torch.float32, device="cuda")
        dc, plans = vdbg.collection_search_device(
            ctx, [(ds, None, None, sg["filter"]) for ds, sg in zip(handles, segs)], 96, "cosine",
            q.data_ptr(), 2, 10, ids.data_ptr(), d.data_ptr(), stream=st.cuda_stream)
    st.synchronize()
    want = oracle.collection_search(segs, 96, "cosine", raw, 10)
    assert np.array_equal(ids.cpu().numpy().view(np.uint64), want[0])
    assert np.array_equal(d.cpu().numpy().view(np.uint32), want[1].view(np.uint32))
    assert np.array_equal(dc, want[2]) and plans == want[3]
    for ds in handles:
        ds.close()


# the largest LDS of each query count (5 queries stage 8 x 816 floats), and one query too many
# for the widest rows (6 x 704 floats are past what the kernel stages)
@pytest.mark.parametrize("dim,counts", [(512, (5, 8)), (768, (5,)), (816, (5,)), (704, (5, 6)),
                                        (1360, (3,)), (2048, (2,))])
def test_small_collection_wide_rows(ctx, oracle, dim, counts):
    segs, handles = build(ctx, [1500, 40, 2100], dim, "cosine", "unit", 700)
    for i, sg in enumerate(segs):
        sg["filter"] = mask(sg["base"].shape[0], 0.4, 80 + i)
    for nq in counts:
        print(f"small collection dim={dim} nq={nq}", flush=True)
        raw = (datagen.clustered_unit(nq, dim, 83, 79, 40, 0.5) * 3).astype(np.float32)
        run(ctx, oracle, segs, handles, dim, "cosine", raw, 10)
    for ds in handles:
        ds.close()


@pytest.mark.parametrize("bad", [np.nan, 0.0])
def test_small_collection_refused_query_writes_nothing(ctx, bad):
    """A NaN or, under cosine, a zero query: the error, and the device results as they were."""
    import torch
    segs, handles = build(ctx, [3000, 2000], 96, "cosine", "unit", 900)
    raw = datagen.clustered_unit(3, 96, 91, 79, 40, 0.5)
    raw[1, :] = bad
    q = torch.from_numpy(raw).cuda()
    ids = torch.full((3, 10), 77, dtype=torch.int64, device="cuda")
    d = torch.full((3, 10), 5.0, dtype=torch.float32, device="cuda")
    with pytest.raises(vdbg.VdbgError) as e:
        vdbg.collection_search_device(ctx, [(ds, None, None, None) for ds in handles], 96,
                                      "cosine", q.data_ptr(), 3, 10, ids.data_ptr(), d.data_ptr())
    assert e.value.code == 1
    torch.cuda.synchronize()
    assert bool((ids == 77).all()) and bool((d == 5.0).all())
    for ds in handles:
        ds.close()


@pytest.mark.parametrize("filt", [None, 0.4, 0.9])
def test_few_queries_over_many_rows(ctx, oracle, filt):
    """Sizes on both sides of the line between one launch over every segment and the lanes (5 to
    8 queries, 6M allowed rows): the same answers."""
    rng = np.random.default_rng(31)
    segs, handles, at = [], [], 0
    for n in (3500000, 3000000):
        base = rng.random((n, 16), dtype=np.float32)
        ds = vdbg.Dataset(ctx, base, 16, "l2")
        ext = np.arange(at, at + n, dtype=np.uint64)
        at += n
        ds.set_external_ids(ext)
        segs.append({"base": base, "ext": ext, "kind": "flat", "deleted": None,
                     "filter": None if filt is None else mask(n, filt, at)})
        handles.append(ds)
    for nq in (4, 8):
        print(f"few queries over many rows nq={nq} filter={filt}", flush=True)
        run(ctx, oracle, segs, handles, 16, "l2", rng.random((nq, 16), dtype=np.float32), 10)
    for ds in handles:
        ds.close()
