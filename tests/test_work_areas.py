"""What the kernels write against what is allocated for it: the launch plans (plans.h, host
arithmetic) enumerated on the CPU, fastmode on panels whose Krylov basis has a lower rank
than its panels have columns, and XTX where its workspace takes several passes."""
import ctypes
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
          // bounded whatever M: 4 GiB of digits and one split's or 2 GiB of sums
          const CodesPlan u = eig_fpca_basis_plan(cu, m, nst, Ct);
          if (F.pa.part_bytes > kFpcaBytes || F.pb.dig_bytes > kFpcaBytes || u.dig_bytes > kFpcaBytes ||
              u.part_bytes > std::max<size_t>(u.part_bytes / u.nsplit, (size_t)2 << 30))
            printf("bounds L=%d I=%d N=%ld M=%ld\n", L, l[1], n, m);
          if (F.arows < 1 || F.arows > m || F.arows > F.pa.rowpad || (F.arows < m && F.arows % 128)) printf("rows L=%d N=%ld M=%ld\n", L, n, m);
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
            const int64_t pmax = cd_max_k(mode) / 128, least = (nblk + pmax - 1) / pmax;
            const int64_t most = smax > least ? smax : least;
            if (P.nsplit > most || P.per > pmax || P.per * P.nsplit < nblk || P.per * (P.nsplit - 1) >= nblk)
              printf("mode %d C %d rows %ld stages %ld smax %d: %d splits of %ld\n", mode, C, nrow, nblk, smax, P.nsplit, P.per);
          }
}
""")
    assert out == []


def test_xtx_workspace_is_bounded(tmp_path):
    # 8 GiB of planes (4,096 SNPs at least) and 4 of sums at every size, bands that cover the
    # tile pairs, and all pairs at once where one pass holds them
    out = run_plans(tmp_path, r"""
int main() {
  for (int64_t n : {1, 128, 129, 198, 1000, 5000, 10184, 17000, 17500, 46000, 85000, 92000, 200000})
    for (int64_t m : {1, 127, 129, 2000, 131073, 600000, 5000000})
      for (int p1 : {7, 8})
        for (int p2 : {6, 7}) {
          const XdPlan X = eig_xd_plan(256, m, (int)((n + 127) / 128), p1, p2);
          const size_t pair = (size_t)X.nsplit * p1 * 256 * 256 * 4, rows = (size_t)X.RT * 32;
          bool ok = X.part_bytes <= kXPartBytes && X.band >= 1 && X.band <= X.npair && X.part_bytes == X.band * pair;
          ok = ok && (X.plane_bytes <= (size_t)kXPlaneBytes || X.K <= 4096) && X.plane_bytes == rows * X.np * X.K;
          ok = ok && X.K % 128 == 0 && X.K <= kXMaxK && X.K * X.nchunk >= m && rows >= (size_t)n;
          ok = ok && X.per % 2 == 0 && (int64_t)X.per * 64 * X.nsplit >= X.K;
          ok = ok && (X.band == X.npair || (X.npair + 0.0) * pair > kXPartBytes);
          if (!ok) printf("N=%ld M=%ld p1=%d p2=%d\n", n, m, p1, p2);
        }
}
""")
    assert out == []


def test_xtx_left_out_parts_cover_a_chunk(tmp_path):
    out = run_plans(tmp_path, r"""
int main() {
  for (int cu : {1, 32, 256})
    for (int64_t n : {2, 129, 257, 2503, 5000, 100000})
      for (int64_t m : {1, 128, 129, 2000, 20011, 131073, 600000}) {
        const int nst = (int)((n + 127) / 128);
        const XdPlan X = eig_xd_plan(cu, m, nst, 7, 6);
        // every SNP is in one split, none of which is empty
        if ((int64_t)X.rsplit * X.rstep * kResSnps < X.K || (int64_t)(X.rsplit - 1) * X.rstep * kResSnps >= X.K) printf("split N=%ld M=%ld\n", n, m);
        // table of 4 pairs a SNP, pairs of each split and of their sum, digit tables
        if (X.tab_bytes < (size_t)X.K * 4 * 16 + (size_t)(X.rsplit + 1) * nst * 128 * 16 + (size_t)X.np * X.K * 4) printf("bytes N=%ld M=%ld\n", n, m);
      }
}
""")
    assert out == []


def test_ranges_of_regrouped_codes_fit_their_area(tmp_path):
    out = run_plans(tmp_path, r"""
int main() {
  for (int C : {1, 10, 11, 16, 20, 21, 64, 240})
    for (int nst : {1, 2, 24, 157, 782, 4000})
      for (int64_t m : {1, 300, 4096, 400000, 600000, 5000000})
        for (int smax : {1, 2, 32}) {
          const int64_t nblk = (m + 127) / 128, nb = eig_codes_chunk(nst, nblk);
          const CodesPlan P = eig_codes_plan(256, kCdSum, C, (int64_t)nst * 128, nblk, smax);
          const CodesPlan Q = eig_codes_plan(256, kCdSum, C, (int64_t)nst * 128, nb, P.nsplit);
          if (nb < 1 || nb > nblk || eig_codes_area(Q) > eig_codes_area(P) || nb > cd_max_k(kCdSum) / 128)
            printf("C=%d nst=%d M=%ld smax=%d\n", C, nst, m, smax);
        }
}
""")
    assert out == []


def test_int32_sums_hold_their_splits(tmp_path):
    # the worst term per code: digit -128 with code 3 (kCdPair), with code 3 and the missing
    # bit's digit (kCdSum), with the missing bit (kCdMiss); -2^31 itself is an INT32
    out = run_plans(tmp_path, r"""
int main() {
  const int64_t term[3] = {128 * 3, 128 * 3 + 128, 128};
  for (int mode = 0; mode < 3; ++mode)
    for (int C : {1, 20, 136})
      for (int64_t nrow : {1, 5000, 200000})
        for (int64_t nblk = 30000; nblk < 90000; nblk += 997)
          for (int smax : {1, 16}) {
            const CodesPlan P = eig_codes_plan(256, mode, C, nrow, nblk, smax);
            if (P.per * 128 * term[mode] > (int64_t)1 << 31) printf("mode %d rows %ld stages %ld\n", mode, nrow, nblk);
          }
}
""")
    assert out == []


@pytest.mark.gpu
def test_xtx_in_bands_of_tile_pairs():
    """17,500 samples: 2,415 tile pairs, two bands of INT32 sums.  The digits' rounding stays
    below FP64's own, so an entry is within M ulps of the largest diagonal entry, as is the
    reference's."""
    import eig_amd
    rng = np.random.default_rng(1)
    N, M = 17500, 200
    g = rng.binomial(2, rng.uniform(0.05, 0.5, M)[:, None], size=(M, N)).astype(np.int32)
    g[rng.random(g.shape) < 0.02] = -1
    print(f"[gpu-case] XTX in bands N={N} M={M}", flush=True)
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        st = eng.snpstats()
        scale, x = eng.xtx(eig_amd.FORM_FP64, 0, want_matrix=True)
    finally:
        eng.close()
    z = (g - st["mean"][:, None]) * st["fancy"][:, None]
    z[(g < 0) | (st["status"] != 0)[:, None]] = 0
    d = (z * z).sum(axis=0)
    y = d.sum() / (N - 1)
    tol = 2 * (M + 16) * 2.0 ** -53 * d.max()
    assert abs(scale - y) <= tol
    worst = 0.0
    for i in range(0, N, 2500):
        ref = z[:, i:i + 2500].T @ z
        worst = max(worst, np.abs(x[i:i + 2500] * scale - ref).max())
    assert worst <= tol


def free():
    """Free and total bytes of the card."""
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value, t.value


def fill(eng, left):
    """Blocks of the card's memory until `left` bytes are free (an allocation may leave more
    free than the count before it had said)."""
    blocks = []
    while (more := free()[0] - left) > 4 << 20:
        blocks.append(eng.dev_alloc(more))
    return blocks


@pytest.mark.gpu
def test_products_without_room_for_the_regrouped_codes():
    """Loadings and FP64 fastmode where the card holds the genotypes and the selection but not
    a third copy of them: ranges of it, the same bits."""
    import eig_amd
    rng = np.random.default_rng(4)
    N, M, K, L = 3000, 400000, 4, 6
    rows = rng.integers(0, 256, (M, N // 4), dtype=np.uint8)
    vec = rng.standard_normal((K, N))
    omega = rng.standard_normal((N, L))
    every, half = np.arange(N, dtype=np.int32), np.arange(N // 2, dtype=np.int32)

    def panel(eng, sel):
        eng.select(sel)
        eng.snpstats(fetch=False)

    def results(eng, n):
        ff, fx = eng.loadings(np.ascontiguousarray(vec[:, :n]))
        ev, v = eng.fpca(2, L, 1, omega=np.ascontiguousarray(omega[:n]))
        return ff, fx, ev, v

    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(rows, N)
        panel(eng, every)
        want = results(eng, N)
    finally:
        eng.close()
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(rows, N)
        panel(eng, every)  # its buffers, and those of the products for half of the samples
        panel(eng, half)
        results(eng, N // 2)
        panel(eng, every)
        # 24 tiles' codes take 307 MB: 154 are there, and 120 more are left free
        blocks = fill(eng, 120 << 20)
        print(f"[gpu-case] regrouped codes in ranges N={N} M={M}", flush=True)
        got = results(eng, N)
        for b in blocks:
            eng.dev_free(b)
    finally:
        eng.close()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.gpu
def test_fastmode_in_passes():
    """1,200,000 SNPs with 64 columns and a basis of 256: X A's sums and X^T U's digits take two
    passes each.  The two leading eigenvalues stand twenty times above the rest, so seven
    products with X and as many with its transpose leave less than 1e-17 of the rest beside
    their axes, and both are XTX's to rounding."""
    import eig_amd
    rng = np.random.default_rng(6)
    N, M, L, I = 300, 1200000, 64, 3
    thr = rng.uniform(0.05, 0.95, (3, M))
    thr = (np.clip(thr, 0.02, 0.98) * 2.0 ** 32).astype(np.uint32)
    pop = np.searchsorted([0.5, 0.8], np.arange(N) / N, side="right").astype(np.int32)
    print(f"[gpu-case] fastmode in passes N={N} M={M}", flush=True)
    eng = eig_amd.Engine(0)
    try:
        eng.synth(M, N, thr, np.repeat(pop[:, None], 3, axis=1), np.full((N, 2), 0xFFFFFFFF, np.uint32),
                  1 << 26, 9)
        eng.select(np.arange(N, dtype=np.int32))
        eng.snpstats(fetch=False)
        scale, _ = eng.xtx(eig_amd.FORM_FP64, 0, want_matrix=False)
        ex, vx = eng.eigh_xtx(3)
        ev, vec = eng.fpca(2, L, I, omega=rng.standard_normal((N, L)))
    finally:
        eng.close()
    want = ex * scale / (2 * M)
    assert want[1] > 20 * want[2]
    assert np.all(np.abs(ev - want[:2]) <= 1e-11 * want[0])
    assert np.max(np.abs(vec - vx[:2])) <= 1e-9


@pytest.mark.gpu
def test_idle_workspaces_are_given_back():
    """An allocation that does not fit frees what XTX and the eigensolver keep between calls;
    their results stay, and the next calls give the same bits."""
    import eig_amd
    rng = np.random.default_rng(2)
    N, M = 700, 30000
    g = rng.binomial(2, rng.uniform(0.05, 0.5, M)[:, None], size=(M, N)).astype(np.int32)
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        eng.snpstats()
        s0, x0 = eng.xtx(eig_amd.FORM_FP64, 0)
        e0, v0 = eng.eigh_xtx(N)
        before, total = free()
        with pytest.raises(eig_amd.EigError):
            eng.dev_alloc(4 * total)
        after, _ = free()
        # 16 planes of 768 samples by 30,000 SNPs alone are 350 MB
        assert after - before >= 300 << 20
        # one that fits once they are gone: 100 MiB free, and 200 to be had
        eng.xtx(eig_amd.FORM_FP64, 0, want_matrix=False)
        blocks = fill(eng, 100 << 20)
        for b in blocks + [eng.dev_alloc(200 << 20)]:
            eng.dev_free(b)
        e1, v1 = eng.eigh_xtx(N)
        s1, x1 = eng.xtx(eig_amd.FORM_FP64, 0)
        e2, v2 = eng.eigh_xtx(N)
    finally:
        eng.close()
    assert s0 == s1 and np.array_equal(x0, x1)
    for e, v in ((e1, v1), (e2, v2)):
        assert np.array_equal(e, e0) and np.array_equal(v, v0)


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
