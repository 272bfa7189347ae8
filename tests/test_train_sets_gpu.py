"""Training on the device: the k-means++ picks (the reference's index-order double sums found in
parallel) against that loop run in numpy on libstdc++'s draws, the sub-quantizers trained all
at once against one at a time, and the encoder against the oracle."""
import numpy as np
import pytest

import vdbg
from ivf_file import parse_pqflat
from vdbg import datagen

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


class Mt64:
    """std::mt19937_64 (the published recurrence), with libstdc++'s uniform_int_distribution
    (Lemire's method on a 64-bit generator) and generate_canonical<double, 53>."""

    def __init__(self, seed):
        self.mt = [seed & M64]
        for i in range(1, 312):
            p = self.mt[-1]
            self.mt.append((6364136223846793005 * (p ^ (p >> 62)) + i) & M64)
        self.i = 312

    def __call__(self):
        mt = self.mt
        if self.i == 312:
            for i in range(312):
                x = (mt[i] & 0xFFFFFFFF80000000) | (mt[(i + 1) % 312] & 0x7FFFFFFF)
                mt[i] = mt[(i + 156) % 312] ^ (x >> 1) ^ (0xB5026F5AA96619E9 if x & 1 else 0)
            self.i = 0
        x = mt[self.i]
        self.i += 1
        x ^= (x >> 29) & 0x5555555555555555
        x ^= (x << 17) & 0x71D67FFFEDA60000
        x ^= (x << 37) & 0xFFF7EEE000000000
        return x ^ (x >> 43)

    def below(self, n):
        p = self() * n
        if (p & M64) < n:
            while (p & M64) < ((1 << 64) - n) % n:
                p = self() * n
        return p >> 64

    def canonical(self):
        r = float(self()) / 2.0 ** 64
        return r if r < 1.0 else np.nextafter(1.0, 0.0)


def l2_any(x, c):
    """L2SqAny of every row: four accumulators over i mod 4, fp32."""
    t = (x - c).astype(np.float32)
    t *= t
    s = [np.zeros(len(x), np.float32) for _ in range(4)]
    d4 = x.shape[1] // 4 * 4
    for i in range(x.shape[1]):
        a = i % 4 if i < d4 else 0
        s[a] = s[a] + t[:, i]
    return (s[0] + s[1]) + (s[2] + s[3])


def pp_picks(x, k, seed):
    rng = Mt64(seed)
    n = len(x)
    cen = [x[rng.below(n)]]
    mind = np.full(n, np.inf, np.float32)
    for _ in range(1, k):
        mind = np.minimum(mind, l2_any(x, cen[-1]))
        acc = np.cumsum(mind.astype(np.float64))  # sequential adds
        if acc[-1] > 0:
            at = np.flatnonzero(acc[:-1] >= rng.canonical() * acc[-1])
            pick = at[0] if at.size else n - 1
        else:
            pick = rng.below(n)
        cen.append(x[pick])
    return np.array(cen)


def points(kind, n, d, seed):
    rng = np.random.default_rng(seed)
    if kind == "int":  # exact sums in any order (the kernel sets' order too)
        return rng.integers(0, 40, (n, d)).astype(np.float32)
    if kind == "uniform":
        return rng.random((n, d), dtype=np.float32)
    if kind == "wide":  # 16 decades: sums round at most points, some halfway
        return (10.0 ** rng.uniform(-8, 8, (n, 1)) * rng.normal(size=(n, d))).astype(np.float32)
    if kind == "grid":  # halves and quarters beside 2^24: ties of the running sum
        return (rng.integers(0, 5, (n, d)) * 0.25 +
                (rng.random((n, 1)) < 0.01) * 2.0 ** 13).astype(np.float32)
    few = rng.random((3, d), dtype=np.float32)  # "few": the total reaches zero
    return few[rng.integers(0, 3, n)]


# (below some 10,000 points of few dims one set is initialised on the host: the sub-quantizers below
# have the device's sets of that size)
# around the tile of 4,096 points; widths with a compiled kernel, without one, and padded ones
# (the kernel sets' distance) up to 128
@pytest.mark.parametrize("n,d,k,kind", [
    (4096, 8, 50, "uniform"), (4097, 4, 50, "wide"), (8191, 8, 60, "wide"),
    (12289, 12, 40, "grid"), (65536, 8, 256, "uniform"), (30000, 3, 100, "wide"),
    (5000, 20, 64, "uniform"), (9000, 16, 64, "int"), (9001, 128, 40, "int"),
    (5000, 8, 16, "few"), (50000, 8, 30, "int"), (4100, 8, 40, "grid")])
def test_kmeanspp_picks(ctx, n, d, k, kind):
    print(f"k-means++ n={n} d={d} k={k} {kind}", flush=True)
    x = points(kind, n, d, 7 * n + d)
    cen, _, _ = vdbg.kmeans(ctx, x, k, iters=0, seed=77, max_points=n, kmeanspp=True)
    want = pp_picks(x, k, 77)
    assert np.array_equal(cen.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,dim,m,kind", [
    (4096, 32, 8, "uniform"), (5003, 96, 8, "wide"), (6000, 40, 8, "int"), (20000, 128, 16, "int"),
    (4500, 64, 4, "int"), (5000, 60, 3, "uniform"), (4097, 64, 16, "wide"), (8191, 64, 8, "wide"),
    (8193, 72, 6, "grid"), (4100, 64, 8, "grid"), (12289, 48, 16, "wide"), (4099, 96, 8, "few"), (4100, 16, 4, "few"), (3000, 32, 8, "uniform")])
def test_sub_quantizers_and_codes(ctx, oracle, n, dim, m, kind):
    """The codebook of a build equals m separate k-means runs (iterations, splits of empty
    clusters and generators included), its codes the oracle's encoder's."""
    print(f"sub-quantizers n={n} dim={dim} m={m} {kind}", flush=True)
    rows = points(kind, n, dim, 3)
    pd = vdbg.padded_dim(dim)
    ds = vdbg.Dataset(ctx, datagen.pad(rows, pd), dim)
    ix = vdbg.PqFlatIndex.build(ds, m, seed=11, max_points=256, iters=5)
    pq = parse_pqflat(ix.save())
    dsub = dim // m
    for j in range(m):
        sub = np.ascontiguousarray(rows[:, j * dsub:(j + 1) * dsub])
        cen, _, _ = vdbg.kmeans(ctx, sub, 256, iters=5, seed=11 + j * 7919, max_points=256)
        got = pq["pq_centroids"].reshape(m, 256, dsub)[j]
        assert np.array_equal(got.view(np.uint32), cen.view(np.uint32)), j
    want = np.empty((n, m), np.uint8)
    for i in range(n):
        oracle.lib.or_pq_encode(pq["pq_centroids"], m, dsub, np.ascontiguousarray(rows[i]), want[i])
    assert np.array_equal(pq["codes"], want)
    ix.close()
    ds.close()
