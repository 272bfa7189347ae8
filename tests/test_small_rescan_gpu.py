"""Small batches without a certificate: the exact re-scan of the chunks that can still hold one
of the answer's rows, queued on the device (device calls) or behind the first read of the results
(host calls, collections), against the oracle.  Rows repeated 60 times, next to each other (few
chunks can hold them) and spread (many can), fail the certificate of every query."""
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


def device_search(ds, qs, k):
    import torch
    q = torch.from_numpy(qs).cuda()
    ids = torch.empty((len(qs), k), dtype=torch.int32, device="cuda")
    d = torch.empty((len(qs), k), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    ds.flat_search_device(q.data_ptr(), len(qs), k, ids.data_ptr(), d.data_ptr())
    ds.ctx.synchronize()
    return ids.cpu().numpy().view(np.uint32), d.cpu().numpy()


def check(got, want):
    assert np.array_equal(got[0], want[1])
    assert np.array_equal(got[1].view(np.uint32), want[0].view(np.uint32))


# the int8 scans of one or two queries and of up to 32 (64, 128 and 256 dims), the row scan over
# fp16 copies, and over fp32 rows at a width with no ranking kernel
@pytest.mark.parametrize("n,dim,nq,k,metric,data", [
    (30000, 128, 1, 10, "l2", "sift"), (30000, 64, 2, 48, "ip", "sift"),
    (100000, 128, 3, 10, "l2", "sift"), (30000, 256, 32, 20, "l2", "sift"),
    (50000, 384, 1, 10, "cosine", "unit"), (20000, 96, 2, 48, "l2", "unit"),
    (9000, 208, 8, 7, "cosine", "unit"), (1100, 400, 5, 10, "l2", "unit")])
@pytest.mark.parametrize("spread", [False, True])
def test_repeated_rows(ctx, oracle, n, dim, nq, k, metric, data, spread):
    print(f"repeated rows n={n} dim={dim} nq={nq} k={k} {metric} spread={spread}", flush=True)
    gen = datagen.sift_like if data == "sift" else (
        lambda c, d, s: datagen.clustered_unit(c, d, s, 213, 40, 0.7))
    base = np.repeat(gen(n // 60 + 1, dim, 211), 60, axis=0)[:n]
    if spread:
        base = base[np.random.default_rng(9).permutation(n)]
    base = np.ascontiguousarray(base)
    qs = gen(nq, dim, 212)
    if nq > 2:  # a query on the rows' outside (no int8 form) and one of huge values (no bound)
        qs[1] += np.float32(0.25)
        qs[2] *= np.float32(1e25)
    ds = vdbg.Dataset(ctx, base, dim, metric)
    rng = np.random.default_rng(n)
    for frac in (None, 0.6, 0.02):
        allow = None if frac is None else words(rng.random(n) < frac)
        want = oracle.flat_search(base, qs, k, metric=metric, allow=allow)
        check(ds.flat_search(qs, k, allow=allow), want)
        if frac is None:
            assert ctx.last_fallbacks() > 0
        try:
            ctx.set_gated_fallbacks(False)
            check(ds.flat_search(qs, k, allow=allow), want)
        finally:
            ctx.set_gated_fallbacks(True)
    check(device_search(ds, qs, k), oracle.flat_search(base, qs, k, metric=metric))
    assert ctx.last_fallbacks() > 0
    ds.close()


@pytest.mark.parametrize("nq,k", [(1, 10), (5, 48)])
def test_repeated_rows_in_some_segments(ctx, oracle, nq, k):
    """Segments with and without repeated rows: those that listed queries are re-scanned."""
    print(f"repeated rows in segments nq={nq} k={k}", flush=True)
    segs, handles, at = [], [], 0
    for i, n in enumerate((4000, 1, 6000, 2500)):
        x = datagen.clustered_unit(n, 96, 220 + i, 229, 40, 0.7)
        if i % 2 == 0:
            x = np.repeat(x[: n // 50], 50, axis=0)
        base = np.ascontiguousarray(x)
        ds = vdbg.Dataset(ctx, base, 96, "cosine")
        ext = np.arange(at, at + n, dtype=np.uint64) * 3
        at += n
        ds.set_external_ids(ext)
        bits = words(np.random.default_rng(i).random(n) < 0.7) if i < 3 else None
        segs.append({"base": base, "ext": ext, "kind": "flat", "deleted": None, "filter": bits})
        handles.append(ds)
    raw = (datagen.clustered_unit(nq, 96, 240, 229, 40, 0.7) * 2).astype(np.float32)
    got = vdbg.collection_search(
        ctx, [(ds, None, None, sg["filter"]) for ds, sg in zip(handles, segs)], 96, "cosine",
        raw, k)
    assert ctx.last_fallbacks() > 0
    want = oracle.collection_search(segs, 96, "cosine", raw, k)
    assert np.array_equal(got[0], want[0])
    assert np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32))
    assert np.array_equal(got[2], want[2]) and got[3] == want[3]
    for ds in handles:
        ds.close()
