"""Split-BF16 fastmode products at the edges of their tiles: SNP counts around the 64-SNP
groups and 128-SNP tiles, sample counts around the 128-sample tiles, panels of 32 and 64
columns, basis products in two chunks and a remainder of one SNP, against the FP64 form with the same start panel.

A value's bf16 hi + lo parts leave at most 2^-17 of it, so a product of two split operands
is off by at most 2^-16 of its terms.  The three population axes stand well apart (their
eigenvalues differ by more than a quarter of the largest), which bounds the eigenvalues'
relative difference by 2^-15 and the eigenvectors' by 2^-12."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,I", [(6, 5), (33, 4)])
@pytest.mark.parametrize("N,M", [(127, 700), (128, 1024), (129, 1025), (257, 639), (384, 1153), (130, 9001)])
def test_split_bf16_panel_edges(N, M, L, I):
    import eig_amd
    rng = np.random.default_rng(N * 31 + M)
    pop = np.searchsorted([0.45, 0.75, 0.92], np.arange(N) / N, side="right")
    p = np.clip(0.5 + 0.25 * rng.standard_normal((4, M)), 0.02, 0.98)
    g = rng.binomial(2, p[pop].T).astype(np.int32)
    g[rng.random(g.shape) < 0.02] = -1
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        eng.snpstats()
        omega = rng.standard_normal((N, L))
        e64, v64 = eng.fpca(2, L, I, omega=omega, form=eig_amd.FORM_FP64)
        e16, v16 = eng.fpca(2, L, I, omega=omega, form=eig_amd.FORM_BF16X4)
    finally:
        eng.close()
    assert np.all(np.abs(e16 - e64) <= 2.0 ** -15 * e64), (e16, e64)
    assert np.max(np.abs(v16 - v64)) <= 2.0 ** -12
