"""Regression windows around the 64 SNPs that one wave decides on, and kept-SNP counts
around its batches of 64 and the chunks of 256, against the oracle.  Bars as in
test_normal_path.py: 1e-10 of the largest entry and of the counts."""
import numpy as np
import pytest

from oracle import oracle as O

from test_normal_path import eng, ld_panel  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ld,M", [(1, 257), (2, 600), (63, 520), (64, 519), (65, 530), (2, 7), (64, 64), (3, 66)])
def test_windows(eng, ld, M):  # noqa: F811
    g, types, chrom, ppos, gpos = ld_panel(31 + M, M, [40, 50, 35])
    N = g.shape[1]
    rows = O.pack_genotypes(g)
    xi = np.arange(N, dtype=np.int32)
    print(f"[gpu-case] ldregress={ld} M={M}", flush=True)
    eng.load_packed(rows, N)
    eng.select(xi)
    eng.snpstats(fetch=False)
    y, yn, st, X = eng.xtx_normal(npop=3, ldregress=ld, chrom=chrom, ppos=ppos, gpos=gpos)
    nc = O.normal_columns(rows, xi, None, None)
    kept = np.nonzero(nc["status"] == 0)[0]
    Z, ynum = O.ldregress_columns(nc["cols"], kept, chrom, ppos, gpos, ld)
    ref, yr = O.dense_xtx(Z)
    assert np.array_equal(st["status"], nc["status"])
    assert abs(y - yr) <= 1e-10 * yr
    assert abs(yn - ynum) <= 1e-10 * ynum
    assert np.max(np.abs(X - ref)) <= 1e-10 * np.max(np.abs(ref))
