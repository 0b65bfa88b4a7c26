"""The FP64 form's XTX (integer digit planes, xdigit.hip) against sums in extended
precision, at the edges of its tiles (256 samples, 32 samples per operand, 64 and 128
SNPs per stage pair) and for panels whose rarest SNP needs more digits.

Tolerance: each of the M products is rounded to the two grids q1 and q2 (p1 and p2
base-256 digits under the power of two above the largest bracket f |x| / 63), the right
integers are at most 126 and 1, so the sum is within M (63 q1 + q2 / 2); the levels and
the final FP64 combination and scaling add a few ulps of the absolute sum.
"""
import math
import sys

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


@pytest.mark.parametrize("N,M,pmin,miss", [
    (2, 1, 0.5, 0.0), (3, 63, 0.2, 0.0), (31, 64, 0.1, 0.1), (33, 65, 0.1, 0.1),
    (127, 128, 0.1, 0.5), (128, 129, 0.1, 0.0), (129, 1000, 0.05, 0.02),
    (255, 300, 0.05, 0.02), (256, 4097, 0.02, 0.02), (257, 2000, 0.001, 0.02),
    (600, 1500, 0.0005, 0.0), (1100, 700, 0.0003, 0.05), (521, 20011, 0.01, 0.02)])
def test_xtx_fp64_against_extended_precision(eng, N, M, pmin, miss):
    rng = np.random.default_rng(N * 7919 + M)
    p = np.exp(rng.uniform(math.log(pmin), math.log(0.5), M))
    g = rng.binomial(2, p[:, None], size=(M, N)).astype(np.int32)
    g[rng.random((M, N)) < miss] = -1
    g[0, :2] = (0, 1)  # the first SNP is kept
    rows = O.pack_genotypes(g)
    xindex = np.arange(N, dtype=np.int32)
    eng.load_packed(rows, N)
    eng.select(xindex)
    st = eng.snpstats()
    print(f"[gpu-case] xtx digits N={N} M={M} pmin={pmin} dropped={int((st['status'] != 0).sum())}",
          flush=True)
    sys.stdout.flush()
    y, mat = eng.xtx(0)
    x = (g - st["mean"][:, None]) * st["fancy"][:, None]
    x[(g < 0) | (st["status"] != 0)[:, None]] = 0.0
    a = float((np.abs(x) * st["fancy"][:, None]).max()) / 63
    E = math.ceil(math.log2(a * 1.01))
    r = 2.0 ** E / math.sqrt(M)
    p1 = 7 if r <= 0.4 else 8
    p2 = 6 if r <= 0.08 else 7
    q1, q2 = 2.0 ** (E + 1 - 8 * p1), 2.0 ** (E + 1 - 8 * p2)
    cols = sorted({0, 1, N // 2, N - 1} | {c for c in (31, 32, 127, 128, 255, 256) if c < N})
    xl = x.astype(np.longdouble)
    want = np.stack([(xl * xl[:, c:c + 1]).sum(axis=0) for c in cols])
    mag = np.stack([(np.abs(x) * np.abs(x[:, c:c + 1])).sum(axis=0) for c in cols])
    got = mat[cols].astype(np.longdouble) * y
    # 16 ulps: f and mu from the levels (4), their products (4), the digits' combination
    # (2), the trace scale and its inverse here (4), and the statistics' own rounding (2)
    tol = M * (63 * q1 + q2 / 2) + 16 * 2.0 ** -53 * mag
    assert np.all(np.abs(got - want) <= tol), float((np.abs(got - want) / tol).max())
    assert np.array_equal(mat, mat.T)
