"""Filtered batches on the ranking GEMMs, whose sample pass reads the filter by sample position
(one bit a sampled row, made with the scan's other start values), against the oracle: samples
below, at and above one 64-bit word, as large as the rows and far smaller; the fp16 and the
int8 GEMM (both of its sample modes); filters that leave all, half, few and no rows."""
import numpy as np
import pytest

import vdbg
from test_row_scan_gpu import check, words
from vdbg import datagen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dim,nq,k,data", [
    (1, 128, 20, 1, "uniform"), (33, 128, 20, 5, "uniform"), (64, 64, 40, 3, "sift"),
    (100, 128, 130, 10, "sift"), (1500, 112, 70, 10, "uniform"), (4097, 128, 300, 10, "sift"),
    (70001, 128, 200, 100, "uniform"), (70001, 128, 2000, 10, "sift"), (9001, 384, 33, 10, "uniform")])
def test_filtered_sample(ctx, oracle, n, dim, nq, k, data):
    print(f"sample filter n={n} dim={dim} nq={nq} k={k} {data}", flush=True)
    make = datagen.sift_like if data == "sift" else datagen.uniform_rows
    base, qs = make(n, dim, 171), make(nq, dim, 172)
    ds = vdbg.Dataset(ctx, base, dim)
    rng = np.random.default_rng(n)
    for frac in (1.0, 0.5, 5.0 / n, 0.0):
        allow = words(rng.random(n) < frac)
        check(ds.flat_search(qs, k, allow=allow), oracle.flat_search(base, qs, k, allow=allow))
    ds.close()
