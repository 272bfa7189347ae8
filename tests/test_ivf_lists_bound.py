"""The bounds of the IVF-PQ scan by list (ivf_lists.hip), checked in float32 on the CPU.

The scan ranks a code of list l for query q by value = offset + fma(-2 2^-(sc + e), sum of fp16(q
2^sc) fp16(r 2^e), rowsum), r the residual its code decodes to, while the reference scores it as
E = offset + sum_j fl(term2[l][j][c_j] + qtab[j][c_j]), four accumulators over j mod 4
(src/index/quant/ivf_pq.cc:203-214).  k_lists_prep claims |value - E| <= eb and |E - |q - c -
r|^2| <= slack, and three rules rest on them:
  - rows of the top R by E have value <= a + 2 eb, a the R-th smallest value of any R rows;
  - a list is left out when (sqrt(offset) (1 - 2^-16) - max |r|)^2 (1 - 2^-20) > T + slack;
  - of the candidates, those with value below a_R - 2 eb belong to the top R by (E, id) and those
    above a_R + 2 eb do not, a_R the R-th smallest value to its upper 20 bits.
numpy float32 operations round each result, so the kernels' and the reference's operation orders
are reproduced here (the matrix unit's order of its sums is not stated: several are tried), over
magnitudes of many binades, queries next to a row (E far below its terms) and rows at the far
edge of their list."""
import numpy as np

F = np.float32
D = np.float64
U = 2.0 ** -24


def dot_any(a, b):
    """Four accumulators over i mod 4, (s0 + s1) + (s2 + s3); the last axis is summed."""
    n = a.shape[-1]
    p = (a * b).astype(F)
    s = [np.zeros(p.shape[:-1], F) for _ in range(4)]
    body = n // 4 * 4
    for i in range(body):
        s[i % 4] = (s[i % 4] + p[..., i]).astype(F)
    for i in range(body, n):
        s[0] = (s[0] + p[..., i]).astype(F)
    return ((s[0] + s[1]).astype(F) + (s[2] + s[3]).astype(F)).astype(F)


def exponent(x):
    """2^e takes the largest magnitude into [2^14, 2^15)."""
    return 15 - int(np.frexp(F(np.abs(x).max()))[1]) if np.abs(x).max() > 0 else 0


def half(x, e, flush):
    h = np.ldexp(x.astype(D), e).astype(np.float16)
    if flush:  # (a unit that takes subnormal halves as zero)
        h = np.where(np.abs(h) < np.float16(2.0 ** -14), np.float16(0), h)
    return h


def sums(p, order, rng):
    """float32 sums over the last axis of exact products p (float64), in one of several orders."""
    n = p.shape[-1]
    if order == "pairs":
        while n > 1:
            p = np.concatenate([(p[..., 0:n - n % 2:2].astype(F) + p[..., 1:n:2].astype(F)).astype(F),
                                p[..., n - n % 2:].astype(F)], axis=-1)
            n = p.shape[-1]
        return p[..., 0].astype(F)
    if order == "blocks":  # 16 exact at a time, added to a float32 accumulator
        acc = np.zeros(p.shape[:-1], F)
        for i in range(0, n, 16):
            acc = (acc + p[..., i:i + 16].sum(-1).astype(F)).astype(F)
        return acc
    if order == "shuffled":
        p = p[..., rng.permutation(n)]
    acc = np.zeros(p.shape[:-1], F)
    for i in range(n):
        acc = (acc + p[..., i].astype(F)).astype(F)
    return acc


class Case:
    """One list and query: the reference's E, the real distances, eb, slack and what they read."""

    def __init__(self, seed, m, dsub, kind):
        rng = self.rng = np.random.default_rng(seed)
        pd, n = m * dsub, 3000
        scale = 10.0 ** rng.uniform(-4, 5)
        cen = rng.standard_normal((m, 256, dsub)) * scale
        if kind == "binades":
            cen *= 2.0 ** rng.integers(-9, 1, (m, 256, dsub))
        cen = cen.astype(F)
        coarse = (rng.standard_normal(pd) * scale * 10.0 ** rng.uniform(-1, 1.5)).astype(F)
        codes = rng.integers(0, 256, (n, m))
        r = cen[np.arange(m), codes].reshape(n, pd)
        far = int(np.argmax((r.astype(D) ** 2).sum(1)))
        if kind == "near":      # next to a row
            q = coarse + r[7] * F(1 + 2.0 ** -12)
        elif kind == "edge":    # behind the list's farthest row
            q = coarse + r[far] * F(rng.choice([1.0, 1.0001, 1.5, 40.0]))
        elif kind == "large":
            q = coarse + rng.standard_normal(pd) * scale * 1e3
        else:
            q = coarse + rng.standard_normal(pd) * scale * (2.0 ** rng.integers(-12, 2, pd)
                                                            if kind == "binades" else 1.0)
        q = q.astype(F)
        # the reference
        t2 = (dot_any(cen, cen) + (F(2) * dot_any(coarse.reshape(m, 1, dsub), cen)).astype(F)).astype(F)
        qt = ((-dot_any(q.reshape(m, 1, dsub), cen)) * F(2)).astype(F)
        diff = (q - coarse).astype(F)
        acc = np.zeros(16, F)
        for i in range(0, pd, 16):
            acc = (acc + (diff[i:i + 16] * diff[i:i + 16]).astype(F)).astype(F)
        self.offset = offset = F(sums(acc.astype(D), "pairs", rng))
        s = [np.zeros(n, F) for _ in range(4)]
        rowsum = np.zeros(n, F)
        for j in range(m):
            s[j % 4] = (s[j % 4] + (t2[j, codes[:, j]] + qt[j, codes[:, j]]).astype(F)).astype(F)
            rowsum = (rowsum + t2[j, codes[:, j]]).astype(F)
        adc = ((s[0] + s[1]).astype(F) + (s[2] + s[3]).astype(F)).astype(F)
        self.E = (offset + adc).astype(F)
        self.real = ((q.astype(D) - coarse.astype(D) - r.astype(D)) ** 2).sum(1)
        # what k_ivf_decode16, IvfMakeDecoded and k_lists_prep keep
        e, sc = exponent(cen), exponent(q)
        norms = np.array([F(sums((r[i:i + 500].astype(D) ** 2), "pairs", rng).max())
                          for i in range(0, n, 500)])
        self.rad = rad = F(np.sqrt(D(norms.max())) * (1 + 1e-4))
        cn = np.sqrt((cen.astype(D) ** 2).sum(2).max(1).sum()) * (1 + 1e-6)
        cc = np.sqrt((coarse.astype(D) ** 2).sum()) * (1 + 1e-6)
        t2abs = D(F(np.abs(t2).max(1).astype(D).sum() * (1 + 2.0 ** -16)))
        nq = np.sqrt(D(F((q.astype(D) ** 2).sum()))) * (1 + 1e-5)
        P = nq * D(rad)
        S = (nq + cc) ** 2 + t2abs + 2 * nq * cn
        sub = 4.0 * pd * 2.0 ** -14 * (np.ldexp(D(np.abs(q).max()), -e) +
                                       np.ldexp(D(np.abs(cen).max()), -sc))
        eb = (2 * P * (2.0 ** -10 + 2.0 ** -21 + (pd + dsub + 32.0) * U) + sub + 2.0 ** -18 * S)
        self.eb = F(eb * 1.001)
        self.slack = F(eb + 2.0 * (pd + 32) * U * ((nq + cc) ** 2 + (cn + cc) ** 2))
        # the values
        flush = bool(rng.integers(0, 2))
        prod = half(q, sc, flush).astype(D) * half(r, e, flush).astype(D)
        order = ("in turn", "pairs", "blocks", "shuffled")[seed % 4]
        dot = sums(prod, order, rng)
        self.v = (np.ldexp(D(-2), -sc - e) * dot.astype(D) + rowsum.astype(D)).astype(F)
        self.value = (offset + self.v).astype(F)


SHAPES = [(16, 8), (4, 32), (8, 2), (16, 3)]
KINDS = ["near", "edge", "large", "binades", "plain"]


def cases():
    for i, (m, dsub) in enumerate(SHAPES):
        for j, kind in enumerate(KINDS):
            for t in range(3):
                yield Case(1000 * i + 10 * j + t, m, dsub, kind)


def enc(f):
    b = f.view(np.uint32)
    return np.where(b & 0x80000000, ~b, b | np.uint32(0x80000000)).astype(np.uint32)


def dec(k):
    k = np.uint32(k)
    return np.uint32(k & 0x7FFFFFFF if k & 0x80000000 else ~k & 0xFFFFFFFF).view(F)


def test_bounds_and_threshold():
    short = 0
    for c in cases():
        err = np.abs(c.value.astype(D) - c.E.astype(D))
        assert (err <= D(c.eb)).all(), (err.max(), c.eb)
        assert (np.abs(c.E.astype(D) - c.real) <= D(c.slack)).all()
        for R in (1, 10, 100):
            top = np.argsort(c.E, kind="stable")[:R]
            # any R rows' R-th smallest value bounds the rest: all rows (the tightest), the first
            for a in (np.sort(c.value)[R - 1], np.sort(c.value[:500])[R - 1]):
                T = F(a + F(2) * c.eb)
                # (the kernel compares v, value without the offset, with T - offset, widened so)
                Td = F(F(T - c.offset) + F(2.0 ** -20) * F(abs(T) + abs(c.offset)))
                assert (c.v[top] <= Td).all()
            short += int((c.value[top] > np.sort(c.value)[R - 1]).any())
    assert short > 0  # the data needs the margin: without it rows of the top R are lost


def test_lists_left_out():
    out = 0
    for c in cases():
        d = F(F(np.sqrt(c.offset)) * F(1 - 2.0 ** -16)) - c.rad
        if not d > 0:
            continue
        low = F(F(F(d) * F(d)) * F(1 - 2.0 ** -20))
        assert D(low) <= c.real.min()
        # thresholds at, just above and just below the scores
        for tau in np.concatenate([np.sort(c.E)[:50], np.nextafter(np.sort(c.E)[:50], F(-np.inf)),
                                   F([c.E.min() * 0.5, 0.0])]):
            if low > F(F(tau) + c.slack):
                out += 1
                assert (c.E > tau).all()
    assert out > 0  # (some list is left out)


def test_sure_members_and_non_members():
    tested = lost = 0
    for c in cases():
        for R in (10, 100):
            for rows in (np.arange(3000), np.argsort(c.value)[:180]):
                val, E = c.value[rows], c.E[rows]
                k = np.sort(enc(val))[R - 1] & ~np.uint32(0xFFF)
                a0, a1 = dec(k), dec(k | np.uint32(0xFFF))
                lo = F(F(a0 - F(2) * c.eb) - F(2.0 ** -20) * F(abs(a0)))
                hi = F(F(a1 + F(2) * c.eb) + F(2.0 ** -20) * F(abs(a1)))
                top = set(np.lexsort((rows, E))[:R].tolist())
                sure = np.flatnonzero(val < lo)
                assert len(sure) <= R and set(sure.tolist()) <= top
                assert not set(np.flatnonzero(val > hi).tolist()) & top
                tested += len(sure)
                first = set(np.argsort(val, kind="stable")[:R].tolist())
                lost += len(top - first)
    assert tested > 0 and lost > 0  # members taken by value alone, and values that misorder


def test_an_eighth_of_the_bound_does_not_hold():
    worst = max((np.abs(c.value.astype(D) - c.E.astype(D)) / D(c.eb)).max() for c in cases())
    assert 0.125 < worst <= 1.0, worst
