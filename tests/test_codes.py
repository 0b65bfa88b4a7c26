"""The products of packed codes with FP64 columns (codes.hip) against sums in extended
precision: loadings (samples summed, two sums per digit set), their scales (SNPs summed,
two digit sets) and lsqproject's normal equations (the missing bits alone), at the edges
of their tiles (16 rows, 128 and 192 to 256 rows a block, 64 and 128 codes a stage, 11 and
20 columns a group) and with a selection that leaves individuals out.

Tolerance: a column's entries are rounded to a grid q = 2^-53 of its largest entry at
most, so a sum of n products with integers up to 3 is within 3 n q / 2 of the exact one
(the three terms of a normalised value: 3 f, 3 f + |l0| and |l0| times that); the final
conversions and factors add a few ulps of the absolute sum.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("nind,M,K,drop,miss", [
    (3, 5, 1, 0, 0.0), (15, 64, 2, 0, 0.2), (17, 65, 3, 1, 0.2), (129, 127, 4, 0, 0.05),
    (130, 129, 10, 2, 0.05), (255, 300, 11, 0, 0.9), (257, 641, 12, 3, 0.05),
    (193, 1000, 16, 0, 0.05), (700, 4100, 10, 50, 0.02)])
def test_code_products_against_extended_precision(eng, nind, M, K, drop, miss):
    rng = np.random.default_rng(nind * 131 + M)
    p = rng.uniform(0.02, 0.5, M)
    g = rng.binomial(2, p[:, None], size=(M, nind)).astype(np.int32)
    g[rng.random((M, nind)) < miss] = -1
    g[0, :3] = (0, 1, 1)
    xindex = np.setdiff1d(np.arange(nind), rng.choice(nind, drop, replace=False)).astype(np.int32)
    n = len(xindex)
    eng.load_packed(O.pack_genotypes(g), nind)
    eng.select(xindex)
    st = eng.snpstats()
    kept = st["status"] == 0
    vec = rng.standard_normal((K, n))
    vec /= np.linalg.norm(vec, axis=1, keepdims=True)
    print(f"[gpu-case] codes nind={nind} M={M} K={K} n={n} kept={int(kept.sum())}", flush=True)
    ff, fx = eng.loadings(vec)
    L = np.longdouble
    mean, fancy = st["mean"].astype(L)[:, None], st["fancy"].astype(L)[:, None]
    x = (g - mean) * fancy
    x[(g < 0) | ~kept[:, None]] = 0
    z = x[:, xindex]
    q = lambda v: 2.0 ** -53 * np.abs(v).max(axis=-1)  # the grid of a column's largest entry
    eps = 2.0 ** -53
    # loadings
    want = 10 * (vec.astype(L) @ z.T)
    mag = 10 * (np.abs(vec) @ np.abs(z).T)
    tol = 10 * 3 * 3 * n * q(vec)[:, None] / 2 * st["fancy"] + 16 * eps * mag
    assert np.all(np.abs(ff - want) <= tol)
    # scales, from the loadings as they came
    f = ff.astype(L)
    fxv = f @ z
    # three terms of up to 3 f |ff| each on a grid of their largest
    qf = q(3 * ff * st["fancy"] * (1 + st["mean"]))
    err = 3 * 3 * M * qf[:, None] / 2 + 16 * eps * (np.abs(ff) @ np.abs(z))
    nrm = np.sqrt((fxv * fxv).sum(axis=1))
    assert np.all(np.abs(1 / fx - nrm) <= np.sqrt((err * err).sum(axis=1)) + (n + 8) * eps * nrm)
    # normal equations of every individual
    use = np.ones(nind, np.int32)
    a, b, s = eng.lsqproject(use, K)
    e = (fx[:, None] * ff).astype(L)
    obs = (g >= 0) & kept[:, None]
    assert np.array_equal(s == 1, obs.sum(axis=0) <= K)
    rhs = e @ x
    qe = q(3 * np.abs(e).astype(float) * st["fancy"] * (1 + st["mean"]))
    tol = 3 * 3 * M * qe[:, None] / 2 + 16 * eps * (np.abs(e) @ np.abs(x))
    ok = s == 0
    assert ok.any() or M < 2 * K
    assert np.all(np.abs(b[:, ok] - rhs[:, ok]) <= tol[:, ok])
    # the solutions satisfy the exact equations to the normal matrices' own rounding:
    # a grid of the largest product of two entries per SNP, and a Cholesky solve's backward
    # error of a few K ulps of the norm
    for i in np.nonzero(ok)[0][:: max(1, ok.sum() // 40)]:
        eo = e[:, obs[:, i]]
        G = eo @ eo.T
        gn = float(np.abs(G).max())
        qg = 2.0 ** -53 * float((np.abs(e).max(axis=1)[:, None] * np.abs(e).max(axis=1)).max())
        dG = M * qg / 2 + 8 * K * K * eps * gn
        r = G @ a[:, i].astype(L) - rhs[:, i]
        assert np.all(np.abs(r) <= K * dG * np.abs(a[:, i]).max() + tol[:, i])
