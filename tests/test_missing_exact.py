"""A missing genotype contributes exactly nothing to a product of codes over SNPs: samples of
which a dozen SNPs are observed keep the accuracy that these dozen give, however many are
missing.

An observed genotype's value is v1 times its code plus v3, both on a grid of at most 2^-53 of
the column's largest |v1|, |v2| or |v3| (v1 = f b, v3 = -xmean b, v2 = (xmean - 3 f) b), so it
is within 3 / 2 of a grid step of the exact one; the sum of n of them is exact up to one
rounding, and the products that make v1 and v3 add a few ulps of each."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
L = np.longdouble
EPS = 2.0 ** -53


def panel(rng, N, M):
    p = rng.uniform(0.05, 0.5, M)
    g = rng.binomial(2, p[:, None], size=(M, N)).astype(np.int32)
    return p, g


def bound(b, st, n):
    """Of the sum over n observed SNPs of b x, b [K, M]: per column."""
    f, xm = st["fancy"], st["mean"] * st["fancy"]
    top = np.abs(b) * np.maximum(np.maximum(f, xm), np.abs(xm - 3 * f))
    return 1.5 * n * EPS * top.max(axis=1)


@pytest.mark.parametrize("M,K", [(4096, 3), (40001, 11)])
def test_sparse_samples_right_hand_sides(M, K):
    import eig_amd
    rng = np.random.default_rng(M)
    N, nobs = 40, K + 8
    p, g = panel(rng, N, M)
    sparse = rng.integers(0, 2, N) == 1
    for i in np.nonzero(sparse)[0]:
        keep = rng.choice(M, nobs, replace=False)
        row = np.full(M, -1, np.int32)
        row[keep] = g[keep, i]
        g[:, i] = row
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        xi = np.nonzero(~sparse)[0].astype(np.int32)
        eng.select(xi)
        st = eng.snpstats()
        kept = st["status"] == 0
        vec = np.linalg.qr(rng.standard_normal((len(xi), K)))[0].T
        print(f"[gpu-case] sparse samples M={M} K={K}", flush=True)
        ff, fx = eng.loadings(np.ascontiguousarray(vec))
        a, b, s = eng.lsqproject(np.ones(N, np.int32), K)
    finally:
        eng.close()
    e = (fx[:, None] * ff).astype(L)
    x = (g - st["mean"].astype(L)[:, None]) * st["fancy"].astype(L)[:, None]
    x[(g < 0) | ~kept[:, None]] = 0
    want = e @ x[:, sparse]
    tol = bound(e.astype(float), st, nobs)[:, None] + 8 * EPS * (np.abs(e) @ np.abs(x[:, sparse]))
    got = b[:, sparse]
    solved = s[sparse] == 0
    assert solved.sum() >= 5
    assert np.all(np.abs(got - want)[:, solved] <= tol[:, solved])


@pytest.mark.parametrize("nq", [5, 40])
def test_sparse_queries_of_the_server(nq):
    """One axis: a coordinate is the right-hand side over the sum of squares, whose products
    are on a grid of their own and which the solve divides by with a few ulps."""
    import eig_amd
    from eig_amd import synth
    rng = np.random.default_rng(nq)
    N, M, nobs = 30, 40001, 9
    p, g = panel(rng, N, M)
    q = np.full((nq, M), 3, np.int32)
    for i in range(nq):
        keep = rng.choice(M, nobs, replace=False)
        q[i, keep] = rng.binomial(2, p[keep])
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        st = eng.snpstats()
        kept = st["status"] == 0
        vec = rng.standard_normal((1, N))
        ff, fx = eng.loadings(vec / np.linalg.norm(vec))
        print(f"[gpu-case] sparse queries nq={nq}", flush=True)
        with eig_amd.Server(eng, nlanes=1) as srv:
            co, stt, _ = srv.poll(srv.submit(synth.pack_samples(q)))
    finally:
        eng.close()
    e = fx[0] * ff[0].astype(L)
    obs = (q < 3) & kept
    x = (q - st["mean"].astype(L)) * st["fancy"].astype(L) * obs
    r, G = x @ e, obs @ (e * e)
    tol = bound(e.astype(float)[None], st, nobs)[0] + 16 * EPS * np.abs(x) @ np.abs(e) + \
        np.abs(r) / G * (nobs * EPS * float(np.abs(e).max()) ** 2 / 2)
    ok = stt == 0
    assert ok.sum() >= 4
    assert np.all(np.abs(co[:, 0] * G - r)[ok] <= tol[ok])
