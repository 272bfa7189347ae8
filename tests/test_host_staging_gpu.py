"""Host calls whose results fill the pinned staging block: the count of uncertified answers goes
out behind them, inside the block."""
import numpy as np
import pytest

import vdbg
from vdbg import datagen

pytestmark = pytest.mark.gpu


# A context's first small call makes a pinned block of 1 MiB; nq x k ids and as many distances
# then take exactly that (32 x 4,096, 16 x 8,192), or one 256-byte step less (31 x 4,228)
@pytest.mark.parametrize("nq,k", [(32, 4096), (16, 8192), (31, 4228)])
@pytest.mark.parametrize("kind", ["flat", "sq8"])
def test_results_of_the_block_size(oracle, nq, k, kind):
    print(f"staged results {kind} nq={nq} k={k}", flush=True)
    n, dim = 9000, 16
    base, qs = datagen.uniform_rows(n, dim, 201), datagen.uniform_rows(nq, dim, 202)
    own = vdbg.Context(0)
    ds = vdbg.Dataset(own, base, dim)
    sq = vdbg.Sq8Index(ds) if kind == "sq8" else None
    # (the second search's results go to the block the first one left)
    for q, kk in ((1, 10), (nq, k)):
        if sq is None:
            ids, d = ds.flat_search(qs[:q], kk)
            od, oi = oracle.flat_search(base, qs[:q], kk)
        else:
            ids, d = sq.search(qs[:q], kk, 0)
            od, oi = oracle.sq8_search(base, sq.codes(), sq.vmin, sq.scale, qs[:q], kk, 0)
        assert np.array_equal(ids, oi)
        assert np.array_equal(d.view(np.uint32), od.view(np.uint32))
    if sq is not None:
        sq.close()
    ds.close()
    own.close()
