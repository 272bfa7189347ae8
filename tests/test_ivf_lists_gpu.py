"""Large IVF-PQ L2 batches, scanned list by list (ivf_lists.hip), against the scan by query over
per-list tables, which scores every row as the reference does: ids, distances and distance
counts must be the same bits.

Sizes stand at the edges of the path: padded dims of every kernel, each code width, lists
shorter and longer than the seeds' 256 slots, tiles with a remainder, the depths of each top-R,
the smallest batch and the batch just below it, scores returned (rerank 0) and re-ranked,
duplicated rows (ties by id; more candidates than a segment holds, scanned by query), and
queries without a bound (huge or NaN components) among ordinary ones."""
import numpy as np
import pytest

import vdbg
from ivf_file import synth_ivfpq
from vdbg import datagen

pytestmark = pytest.mark.gpu


def _rows(n, dim, seed):
    v = datagen.sift_like(n, dim, seed)
    return np.ascontiguousarray(np.pad(v, ((0, 0), (0, -dim % 16))))


def _same(ctx, ix, qs, k, nprobe, rerank):
    ctx.set_ivf_row_sums(False)
    try:
        ri, rd, rc = ix.search(qs, k, nprobe, rerank)
    finally:
        ctx.set_ivf_row_sums(True)
    gi, gd, gc = ix.search(qs, k, nprobe, rerank)
    assert np.array_equal(gc, rc)
    assert np.array_equal(gd.view(np.uint32), rd.view(np.uint32))
    assert np.array_equal(gi, ri)


def _fewest(n, nlist, nprobe):
    """The smallest batch the scan by list takes."""
    return int(np.ceil((12e6 + 50.0 * n) / (nprobe * n / nlist)))


@pytest.mark.parametrize("n,dim,nlist,m,nprobe,rerank,k,more", [
    (20000, 128, 64, 16, 8, 100, 10, 0),      # the smallest batch
    (20000, 128, 64, 16, 8, 100, 10, -1),     # one query below: the scan by query
    (20000, 128, 64, 16, 8, 0, 10, 1),        # scores returned
    (20000, 16, 64, 4, 16, 100, 10, 127),
    (20000, 24, 64, 8, 64, 64, 1, 1),         # every list probed, padding in the rows
    (12000, 48, 61, 16, 9, 65, 7, 5),
    (12000, 64, 64, 4, 7, 128, 10, 0),
    (9000, 80, 100, 8, 30, 129, 100, 63),
    (9000, 96, 300, 16, 100, -1, 25, 3),      # lists of 30 rows
    (9000, 112, 64, 4, 16, 256, 10, 2),       # the deepest
    (60000, 32, 16, 8, 12, 100, 100, 1),      # lists of 3,750 rows: minima of 4
    (3000, 32, 4, 8, 4, 100, 10, 0),          # as many lists as give seeds
])
def test_list_scan_is_the_scan_by_query(ctx, n, dim, nlist, m, nprobe, rerank, k, more):
    nq = _fewest(n, nlist, nprobe) + more
    print(f"ivf lists {n}x{dim} nlist={nlist} m={m} nq={nq} nprobe={nprobe} {rerank} {k}",
          flush=True)
    base = _rows(n, dim, 4101)
    qs = _rows(nq, dim, 4102)
    ix = vdbg.IvfPqIndex.load(vdbg.Dataset(ctx, base, dim), synth_ivfpq(base, dim, nlist, m, seed=7))
    _same(ctx, ix, qs, k, nprobe, rerank)


# the compiled code widths that the sizes above leave out, scores returned and re-ranked
@pytest.mark.parametrize("dim,m", [(64, 16), (128, 8), (96, 8), (64, 8), (128, 4), (96, 4), (32, 4)])
def test_list_scan_code_widths(ctx, dim, m):
    n, nlist, nprobe = 20000, 64, 8
    nq = _fewest(n, nlist, nprobe)
    print(f"ivf lists widths {dim} m={m} nq={nq}", flush=True)
    base = _rows(n, dim, 4101)
    qs = _rows(nq, dim, 4102)
    ix = vdbg.IvfPqIndex.load(vdbg.Dataset(ctx, base, dim), synth_ivfpq(base, dim, nlist, m, seed=7))
    _same(ctx, ix, qs, 10, nprobe, 100)
    _same(ctx, ix, qs, 150, nprobe, 0)


@pytest.mark.parametrize("nq,nprobe", [(65600, 8), (62000, 256)])
def test_list_scan_in_passes(ctx, nq, nprobe):
    """More queries than a pass takes: 65,536, or fewer with many probes a query (its scratch)."""
    n, dim, nlist = 20000, 16, 256
    print(f"ivf lists passes nq={nq} nprobe={nprobe}", flush=True)
    base, qs = _rows(n, dim, 4121), _rows(nq, dim, 4122)
    ix = vdbg.IvfPqIndex.load(vdbg.Dataset(ctx, base, dim), synth_ivfpq(base, dim, nlist, 4, seed=9))
    _same(ctx, ix, qs, 10, nprobe, 20)


def test_list_scan_duplicates_and_unbounded_queries(ctx):
    print("ivf lists duplicated rows, huge and NaN queries", flush=True)
    uniq = (datagen.sift_like(1500, 64, 4111) - 60.0).astype(np.float32) * np.float32(0.013)
    base = np.ascontiguousarray(np.tile(uniq, (12, 1)))
    qs = np.concatenate([uniq[:1000], uniq[:1000] * np.float32(1e-25)])
    qs[3] *= np.float32(1e21)
    qs[77, 5] = np.nan
    qs[78] = 0.0
    qs[79] *= np.float32(1e-44)
    qs[1500] = np.inf
    ix = vdbg.IvfPqIndex.load(vdbg.Dataset(ctx, base, 64), synth_ivfpq(base, 64, 40, 16, seed=8))
    for rerank, k in [(100, 10), (0, 100)]:
        ctx.set_ivf_row_sums(False)
        ri, rd, rc = ix.search(qs, k, 20, rerank)
        ctx.set_ivf_row_sums(True)
        gi, gd, gc = ix.search(qs, k, 20, rerank)
        ok = np.isfinite(qs).all(axis=1)  # (answers of queries without finite distances are open)
        assert np.array_equal(gi[ok], ri[ok])
        assert np.array_equal(gd[ok].view(np.uint32), rd[ok].view(np.uint32))
        assert np.array_equal(gc[ok], rc[ok])
