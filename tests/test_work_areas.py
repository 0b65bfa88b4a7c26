"""What the kernels write against what is allocated for it: the launch plans (plans.h, host
arithmetic) enumerated on the CPU, and fastmode on panels whose Krylov basis has a lower rank
than its panels have columns."""
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eig_amd", "csrc")


def run_plans(tmp_path, body):
    """Lines that a program around plans.h prints."""
    src, exe = tmp_path / "plans.cpp", tmp_path / "plans"
    src.write_text('#include <cstdio>\n#include "plans.h"\n' + body)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    return subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()


def test_fastmode_area_holds_every_rank(tmp_path):
    # panels of one column to the 256 that a basis may have, tiles from one to many rounds of blocks
    out = run_plans(tmp_path, r"""
int main() {
  const int li[][2] = {{30, 7}, {21, 10}, {20, 10}, {11, 1}, {20, 5}, {40, 5}, {3, 1}, {128, 1}};
  const int64_t ns[] = {1, 129, 200, 256, 1000, 4050, 4100, 4200, 4300, 17500, 100000};
  const int64_t ms[] = {1, 15, 40, 130, 215, 600, 2000, 20000, 100000, 500000, 9000000};
  for (auto &l : li)
    for (int64_t n : ns)
      for (int64_t m : ms)
        for (int cu : {32, 256}) {
          const int L = l[0], Ct = (l[1] + 1) * L, nst = (int)((n + 127) / 128);
          const FpcaPlans F = eig_fpca_plans(cu, m, nst, 1, L, Ct);
          if (eig_codes_area(F.pa) > F.area || eig_codes_area(F.pb) > F.area) printf("panel L=%d N=%ld M=%ld\n", L, n, m);
          for (int r = 1; r <= Ct; ++r)
            if (eig_codes_area(eig_fpca_basis_plan(cu, m, nst, r)) > F.area) printf("L=%d I=%d N=%ld M=%ld r=%d\n", L, l[1], n, m, r);
        }
}
""")
    assert out == []


def test_plan_keeps_its_split_bound(tmp_path):
    out = run_plans(tmp_path, r"""
int main() {
  for (int mode = 0; mode < 3; ++mode)
    for (int C : {1, 11, 12, 20, 21, 55, 136, 240})
      for (int64_t nrow : {1, 64, 193, 5000, 600000})
        for (int64_t nblk : {1, 2, 3, 7, 40, 157, 4688, 40960, 40961, 100000})
          for (int smax : {1, 2, 5, 32, 512}) {
            const CodesPlan P = eig_codes_plan(256, mode, C, nrow, nblk, smax);
            const int64_t pmax = kCodesMaxK / 128, least = (nblk + pmax - 1) / pmax;
            const int64_t most = smax > least ? smax : least;
            if (P.nsplit > most || P.per > pmax || P.per * P.nsplit < nblk || P.per * (P.nsplit - 1) >= nblk)
              printf("mode %d C %d rows %ld stages %ld smax %d: %d splits of %ld\n", mode, C, nrow, nblk, smax, P.nsplit, P.per);
          }
}
""")
    assert out == []


@pytest.mark.gpu
@pytest.mark.parametrize("N,M,L,I", [(200, 15, 11, 1), (4200, 215, 30, 7)])
def test_fastmode_basis_of_lower_rank(N, M, L, I):
    """M < (I + 1) L: the basis spans all of the SNPs' space, so the eigenpairs are the
    panel's own.  The products round at 2^-53 of their columns' largest entries and the basis
    is orthonormal to some 100 ulps, so 1e-11 of the largest eigenvalue covers the
    eigenvalues, and over the gaps (5 per cent of it at least: three axes of four
    populations stand apart) 1e-9 the eigenvectors."""
    import eig_amd
    rng = np.random.default_rng(N + M)
    pop = np.searchsorted([0.45, 0.75, 0.92], np.arange(N) / N, side="right")
    p = np.clip(0.5 + 0.3 * rng.standard_normal((4, M)), 0.02, 0.98)
    g = rng.binomial(2, p[pop].T).astype(np.int32)
    g[rng.random(g.shape) < 0.02] = -1
    print(f"[gpu-case] fastmode rank {M} of {(I + 1) * L}, N={N}", flush=True)
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        st = eng.snpstats()
        ev, vec = eng.fpca(2, L, I, omega=rng.standard_normal((N, L)))
    finally:
        eng.close()
    x = (g - st["mean"][:, None]) * st["fancy"][:, None] / np.sqrt(2.0)
    x[g < 0] = 0
    _, s, vt = np.linalg.svd(x, full_matrices=False)
    want = s ** 2 / M
    gap = min(want[0] - want[1], want[1] - want[2])
    assert gap > 0.05 * want[0]
    assert np.all(np.abs(ev - want[:2]) <= 1e-11 * want[0])
    v = vt[:2] * np.sign(vt[:2][np.arange(2), np.abs(vt[:2]).argmax(axis=1)])[:, None]
    assert np.max(np.abs(vec - v)) <= 1e-9
