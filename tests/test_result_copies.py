"""Results of every size that reaches the host by its own route: up to 128 KB together, up
to 2 MB alone, and beyond in 1 MB pieces by several threads.  Statistics are whole numbers
and single roundings; a loading is a sum of N products, off by at most (N + 4) 2^-53 of the
sum of their magnitudes."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 32767, 32768, 32769, 65537, 262143, 262144, 262145, 393217, 1048577])
def test_sizes(M):
    import eig_amd
    N, K = 8, 2
    rng = np.random.default_rng(M)
    g = rng.integers(0, 3, (M, N)).astype(np.int32)
    g[:, 0], g[:, 1] = 0, 2  # both alleles seen: every SNP is kept
    v = rng.standard_normal((K, N))
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        for _ in range(2):
            st = eng.snpstats()
            ff, fx = eng.loadings(v)
        assert eng.last_ms("snpstats") > 0 and eng.last_ms("loadings") > 0
        assert eng.last_ms("no such stage") == -1
    finally:
        eng.close()
    assert np.array_equal(st["c0"], g.sum(1)) and not st["nmiss"].any() and not st["status"].any()
    mean = g.sum(1) / N
    assert np.array_equal(st["mean"], mean)
    p = 0.5 * mean
    assert np.allclose(st["fancy"], 1 / np.sqrt(p * (1 - p)), rtol=4 * 2.0 ** -53, atol=0)
    z = (g - mean[:, None]) * st["fancy"][:, None]
    bound = 10 * (N + 4) * 2.0 ** -53 * (np.abs(v) @ np.abs(z).T)
    assert np.all(np.abs(ff - 10 * (v @ z.T)) <= bound)
