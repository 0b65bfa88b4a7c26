// SNP loadings, projection scales and lsqproject on the device.
//
//  loadings : ffvecs[j][m] = sum_i 10 v_j[i] z_m[i], a product of the samples' codes with
//             the axes (codes.hip).
//  fxscal   : fxvecs[j][i] = sum_m x_i[m] ffvecs[j][m] with the reference's row
//             fix-up x = g*fancy - mean*fancy (missing or ignored -> 0), a product of
//             the SNPs' codes with the loadings.
//  lsqproject: per individual, over observed SNPs, the K x K Gram of
//             e_m = fxscal .* ffvecs[:,m] and the right-hand side sum_m e_m x_m, as
//             products of the codes and the missing bits with the e_m e_m^T and e_m (with
//             usepopsformissing's fill: FP64 sums over fixed SNP chunks in chunk order),
//             then the Cholesky solve of nicksrc/linsubs.c (choldc/cholsl) per individual.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "eig_internal.h"

constexpr int kLsqChunk = 4096;  // SNPs per lsqproject partial

// run the statement with the compile-time constant KC equal to the runtime K (1..16)
#define EIG_KCASE(n, ...) \
  case n: {               \
    constexpr int KC = n; \
    __VA_ARGS__;          \
  } break;
#define EIG_KSWITCH(k, ...)                                                                  \
  switch (k) {                                                                               \
    EIG_KCASE(1, __VA_ARGS__) EIG_KCASE(2, __VA_ARGS__) EIG_KCASE(3, __VA_ARGS__)             \
    EIG_KCASE(4, __VA_ARGS__) EIG_KCASE(5, __VA_ARGS__) EIG_KCASE(6, __VA_ARGS__)             \
    EIG_KCASE(7, __VA_ARGS__) EIG_KCASE(8, __VA_ARGS__) EIG_KCASE(9, __VA_ARGS__)             \
    EIG_KCASE(10, __VA_ARGS__) EIG_KCASE(11, __VA_ARGS__) EIG_KCASE(12, __VA_ARGS__)          \
    EIG_KCASE(13, __VA_ARGS__) EIG_KCASE(14, __VA_ARGS__) EIG_KCASE(15, __VA_ARGS__)          \
    EIG_KCASE(16, __VA_ARGS__)                                                                \
    default:                                                                                 \
      return eig_set_err(ctx, EIG_E_ARG, "K out of range");                                  \
  }

// ---------------------------------------------------------------- loadings
// ignore[m] (status not kept, unless the caller gave a mask) and xmean = mean * fancy
__global__ void k_load_prep(const int32_t *__restrict__ status, const double *__restrict__ mean,
                            const double *__restrict__ fancy, int64_t M, int32_t mask,
                            uint8_t *__restrict__ ignore, double *__restrict__ xmean) {
  const int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (m >= M) return;
  if (mask) ignore[m] = status[m] != EIG_SNP_KEPT;
  xmean[m] = mean[m] * fancy[m];
}

// fxscal[j] = 1 / sqrt(sum_i fxvecs[j][i]^2)
__global__ void k_fxscal(const double *__restrict__ fxvecs, int32_t nrows,
                         double *__restrict__ fxscal) {
  __shared__ double red[256];
  const int j = blockIdx.x;
  double s2 = 0.0;
  for (int32_t i = threadIdx.x; i < nrows; i += 256) {
    const double s = fxvecs[(int64_t)j * nrows + i];
    s2 += s * s;
  }
  red[threadIdx.x] = s2;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) fxscal[j] = 1.0 / sqrt(red[0]);
}

// ---------------------------------------------------------------- lsqproject
// Individuals read from GENO rows (all loaded samples).  Per (individual block of
// 64, SNP chunk): Gram upper triangle (K(K+1)/2), rhs (K), observed count.
template <int K>
__global__ __launch_bounds__(64) void k_lsq_gram(const uint8_t *__restrict__ geno, int64_t rlen,
                                                 int64_t M, int32_t nind,
                                                 const double *__restrict__ ff,
                                                 const double *__restrict__ fxscal,
                                                 const double *__restrict__ fancy,
                                                 const double *__restrict__ xmean,
                                                 const uint8_t *__restrict__ ignore,
                                                 const double *__restrict__ fill,
                                                 const int32_t *__restrict__ itype, int32_t npop,
                                                 double *__restrict__ partial, int32_t nblk) {
  __shared__ double se[64][kMaxK + 2];
  const int li = threadIdx.x;
  const int32_t q = (blockIdx.x % nblk) * 64 + li;
  const int64_t chunk = blockIdx.x / nblk;
  const int64_t m0 = chunk * kLsqChunk, m1 = min(M, m0 + kLsqChunk);
  constexpr int nP = K * (K + 1) / 2;
  double G[nP];
  double r[K];
#pragma unroll
  for (int p = 0; p < nP; ++p) G[p] = 0.0;
#pragma unroll
  for (int j = 0; j < K; ++j) r[j] = 0.0;
  double kk = 0.0, nobs = 0.0;
  const int32_t ty = q < nind ? itype[q] : -1;
  for (int64_t mb = m0; mb < m1; mb += 64) {
    __syncthreads();
    {
      int64_t m = mb + li;
      bool ok = m < m1;
#pragma unroll
      for (int j = 0; j < K; ++j) se[li][j] = ok ? fxscal[j] * ff[(int64_t)j * M + m] : 0.0;
      se[li][K] = ok ? (ignore[m] ? -1.0 : fancy[m]) : -1.0;
      se[li][K + 1] = ok ? xmean[m] : 0.0;
    }
    __syncthreads();
    const int64_t lim = min((int64_t)64, m1 - mb);
    if (q < nind) {
      for (int rr = 0; rr < lim; ++rr) {
        double fz = se[rr][K];
        if (fz < 0.0) continue;  // ignored SNP: reads as missing
        uint32_t b = geno[(mb + rr) * rlen + (q >> 2)];
        uint32_t code = (b >> ((3 - (q & 3)) << 1)) & 3u;
        double gv = (double)code;
        if (code == 3u) {
          // usepopsformissing: the mean genotype of the individual's population type
          // (lsqproj, smartpca.c:4680-4690); without one the SNP is unobserved
          if (ty < 0) continue;
          gv = fill[(mb + rr) * npop + ty];
          if (isnan(gv)) continue;
        } else {
          nobs += 1.0;
        }
        double x = gv * fz;
        x = (x < -0.001) ? 0.0 : x - se[rr][K + 1];
        kk += 1.0;
        double e[K];
#pragma unroll
        for (int a = 0; a < K; ++a) e[a] = se[rr][a];
#pragma unroll
        for (int a = 0; a < K; ++a) r[a] += e[a] * x;
#pragma unroll
        for (int a = 0; a < K; ++a)
#pragma unroll
          for (int c = a; c < K; ++c) G[a * K - a * (a - 1) / 2 + (c - a)] += e[a] * e[c];
      }
    }
  }
  if (q < nind) {
    double *out = partial + (chunk * (int64_t)nind + q) * (nP + K + 2);
#pragma unroll
    for (int p = 0; p < nP; ++p) out[p] = G[p];
#pragma unroll
    for (int j = 0; j < K; ++j) out[nP + j] = r[j];
    out[nP + K] = kk;
    out[nP + K + 1] = nobs;
  }
}

// reduce chunks in order, Cholesky solve (choldc/cholsl order of operations)
// itype (may be NULL): with the fill, an individual of type >= 0 is also ignored when
// its observed genotypes alone number <= K (lsqproj's first loop, smartpca.c:4637-4651).
template <int K>
__global__ __launch_bounds__(64) void k_lsq_solve(const double *__restrict__ partial, int64_t nchunk,
                                                  int32_t nind, const int32_t *__restrict__ use,
                                                  const int32_t *__restrict__ itype,
                                                  double *__restrict__ ans, double *__restrict__ rhs_out,
                                                  int32_t *__restrict__ st) {
  const int32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nind) return;
  constexpr int nP = K * (K + 1) / 2, W = nP + K + 2;
  double acc[W];
#pragma unroll
  for (int p = 0; p < W; ++p) acc[p] = 0.0;
  for (int64_t c = 0; c < nchunk; ++c) {
    const double *pp = partial + (c * (int64_t)nind + q) * W;
#pragma unroll
    for (int p = 0; p < W; ++p) acc[p] += pp[p];
  }
#pragma unroll
  for (int j = 0; j < K; ++j) rhs_out[(int64_t)j * nind + q] = acc[nP + j];
  if (!use[q]) {
    st[q] = 3;
    return;
  }
  if (acc[nP + K] <= (double)K || (itype && itype[q] >= 0 && acc[nP + K + 1] <= (double)K)) {
    st[q] = 1;
    return;
  }
  // the upper triangle at (i, j), j >= i, holds a[i][j] until step (i, j) puts the factor's
  // [j][i] there: constant indices, so everything stays in registers
  auto at = [&](int i, int j) -> double & { return acc[i * K - i * (i - 1) / 2 + (j - i)]; };
  double p[K], x[K];
  bool bad = false;
#pragma unroll
  for (int i = 0; i < nP + K; ++i) bad |= isnan(acc[i]);
#pragma unroll
  for (int i = 0; i < K; ++i) {
#pragma unroll
    for (int j = i; j < K; ++j) {
      double s = at(i, j);
#pragma unroll
      for (int k = i - 1; k >= 0; --k) s -= at(k, i) * at(k, j);
      if (i == j) {
        bad |= s <= 0.0;
        p[i] = sqrt(s > 0.0 ? s : 1.0);
      } else {
        at(i, j) = s / p[i];
      }
    }
  }
  if (bad) {
    st[q] = 2;
    return;
  }
#pragma unroll
  for (int i = 0; i < K; ++i) {
    double s = acc[nP + i];
#pragma unroll
    for (int k = i - 1; k >= 0; --k) s -= at(k, i) * x[k];
    x[i] = s / p[i];
  }
#pragma unroll
  for (int i = K - 1; i >= 0; --i) {
    double s = x[i];
#pragma unroll
    for (int k = i + 1; k < K; ++k) s -= at(i, k) * x[k];
    x[i] = s / p[i];
  }
#pragma unroll
  for (int j = 0; j < K; ++j) ans[(int64_t)j * nind + q] = x[j];
  st[q] = 0;
}

extern "C" int eig_loadings(eig_ctx *ctx, const double *evecs, int32_t K, const uint8_t *ignore,
                            double *ffvecs, double *fxscal) {
  if (!ctx || !evecs || K <= 0 || K > kMaxK)
    return eig_set_err(ctx, EIG_E_ARG, "eig_loadings: K must be in [1, %d]", kMaxK);
  if (!ctx->have_stats) return eig_set_err(ctx, EIG_E_STATE, "eig_loadings before eig_snpstats");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  const int64_t M = ctx->nsnp;
  const int32_t n = ctx->nrows;
  hipStream_t st = ctx->stream;
  EIG_TRY(eig_ensure(ctx, ctx->ignore_dev, M));
  EIG_TRY(eig_ensure(ctx, ctx->ffvecs, 8 * (size_t)K * M));
  EIG_TRY(eig_ensure(ctx, ctx->fxscal, 8 * (size_t)(kMaxK + M)));  // fxscal | xmean
  EIG_TRY(eig_ensure(ctx, ctx->projw, 8 * (size_t)K * n * 2));     // axes | fxvecs
  // without room for the regrouped codes the product over SNPs takes ranges of them
  const int rg = eig_ensure_selg(ctx);
  if (rg != EIG_OK && rg != EIG_E_NOMEM) return rg;
  double *d_fx = (double *)ctx->fxscal.p, *d_xm = d_fx + kMaxK;
  double *d_ev = (double *)ctx->projw.p, *d_fxv = d_ev + (size_t)K * n;
  double *d_ff = (double *)ctx->ffvecs.p;
  uint8_t *d_ign = (uint8_t *)ctx->ignore_dev.p;
  if (ignore) EIG_HIP(ctx, hipMemcpyAsync(d_ign, ignore, M, hipMemcpyHostToDevice, st));
  EIG_HIP(ctx, hipMemcpyAsync(d_ev, evecs, 8 * (size_t)K * n, hipMemcpyHostToDevice, st));
  // ffvecs = 10 Z^T v as a product over the samples (rows = SNPs), fxvecs = X ff as one
  // over the SNPs (rows = samples), on the code planes (codes.hip).  At 5,000 x 600,000,
  // K = 10, both read the codes once: 19.6 ms with per-code bins and FP64 sums on the
  // vector units, 1.45 now.
  const CodeView vm{(const uint8_t *)ctx->sel.p, nullptr, 128 * 32, 32, M * 32, 16, M,
                    (int64_t)ctx->nst * 8, kCodeLinear};
  CodeCols ax{kColAxes, d_ev, n, n};
  CodeCols fc{kColFx, d_ff, M, M};
  fc.fancy = (const double *)ctx->fancy.p;
  fc.xmean = d_xm;
  fc.ignore = d_ign;
  const CodesPlan pl = eig_codes_plan(ctx->num_cu, kCdPair, K, M, ctx->nst, 16);
  const CodesPlan pf = eig_codes_plan(ctx->num_cu, kCdSum, K, (int64_t)ctx->nst * kTileS, (M + 127) / 128, 32);
  EIG_TRY(eig_ensure(ctx, ctx->scratch2, std::max(eig_codes_area(pl), eig_codes_area(pf))));
  char *ws = (char *)ctx->scratch2.p;
  eig_time_begin(ctx);
  hipLaunchKernelGGL(k_load_prep, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, st,
                     (const int32_t *)ctx->status.p, (const double *)ctx->mean.p,
                     (const double *)ctx->fancy.p, M, ignore ? 0 : 1, d_ign, d_xm);
  EIG_TRY(eig_codes_scales(ctx, pl, ax, ws, st));
  EIG_TRY(eig_codes_mul(ctx, pl, vm, ax, 0, ws, ws + pl.head_bytes, ws + pl.head_bytes + pl.dig_bytes,
                        false, st));
  EIG_TRY(eig_codes_out_pair(ctx, pl, M, ws, ws + pl.head_bytes + pl.dig_bytes,
                             (const double *)ctx->lev.p, d_ign, 10.0, d_ff, 1, M, st));
  EIG_TRY(eig_codes_samples(ctx, pf, fc, ws, n, 1.0, d_fxv, 1, n, K, st));
  hipLaunchKernelGGL(k_fxscal, dim3((unsigned)K), dim3(256), 0, st, (const double *)d_fxv, n, d_fx);
  EIG_HIP(ctx, hipGetLastError());
  eig_time_end(ctx, "loadings");
  EigFetch f(ctx);
  EIG_TRY(f.get(ffvecs, ctx->ffvecs.p, 8 * (size_t)K * M));
  EIG_TRY(f.get(fxscal, d_fx, 8 * (size_t)K));
  EIG_TRY(f.wait());
  ctx->last_K = K;
  ctx->have_load = true;
  return EIG_OK;
}

// ---------------------------------------------------------------- normal equations
// GENO rows of SNPs m0 .. (64 per group) and individuals q0 .. (128 per tile) as the
// grouped codes of eig_ensure_selg: 16 bytes per (tile, group, individual).  SNPs past M
// and individuals past nind read as missing.
__global__ __launch_bounds__(256) void k_regroup_geno(const uint8_t *__restrict__ geno, int64_t rlen,
                                                      int64_t M, int32_t nind, int64_t m0, int32_t q0,
                                                      int64_t G64, int64_t ngroups,
                                                      uint4 *__restrict__ out) {
  __shared__ __align__(4) uint8_t by[2][kGrp][36];
  const int half = threadIdx.x >> 7, i = threadIdx.x & 127;
  const int64_t gid = (int64_t)blockIdx.x * 2 + half;  // tile * G64 + group
  const bool live = gid < ngroups;
  const int64_t tile = live ? gid / G64 : 0, g = live ? gid % G64 : 0;
  const int64_t b0 = q0 / 4 + tile * 32;  // first byte of the tile's 128 individuals
  const int64_t nby = (nind + 3) / 4;
  // four bytes a load (rows start at any byte; the hardware takes unaligned words), single
  // ones where a row's last word would pass its end
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int idx = i + 128 * e, r = idx >> 3, b = (idx & 7) * 4;
    const int64_t m = m0 + g * kGrp + r;
    const uint8_t *src = geno + m * rlen + b0 + b;
    uint32_t word = ~0u;
    if (live && m < M) {
      if (b0 + b + 4 <= nby) {
        __builtin_memcpy(&word, src, 4);
      } else {
        for (int u = 0; u < 4; ++u)
          if (b0 + b + u < nby) word = (word & ~(0xFFu << (8 * u))) | ((uint32_t)src[u] << (8 * u));
      }
    }
    *(uint32_t *)&by[half][r][b] = word;
  }
  __syncthreads();
  if (!live) return;
  const bool in = q0 + tile * 128 + i < nind;
  const int sh = 6 - 2 * (i & 3);
  uint32_t o[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t c = ((uint32_t)by[half][16 * s + 8 * h + j][i >> 2] >> sh) & 3u;
        o[2 * h + (s >> 1)] |= c << (16 * (s & 1) + 2 * j);
      }
  out[gid * kTileS + i] = in ? make_uint4(o[0], o[1], o[2], o[3]) : make_uint4(~0u, ~0u, ~0u, ~0u);
}

// The normal equations of every individual, acc[q][W]: the Gram's upper triangle, the
// right-hand side and the observed count, from the current loadings, in a workspace of
// `bytes` at ws.  The Gram is the sum of e e^T over all kept SNPs minus that over the
// individual's missing ones, so it needs the missing bits alone.  Individuals run in
// chunks of whole tiles and SNPs in chunks of whole stages, as the workspace holds; the
// sums within kLsqRange stages are exact, so the chunks do not change the result.
constexpr int64_t kLsqRange = ((int64_t)5 << 20) / 128 / 2;  // below cd_max_k of both products
static int lsq_normal(eig_ctx *ctx, double *acc, char *ws, size_t bytes) {
  const int64_t M = ctx->nsnp;
  const int32_t nind = ctx->nind, K = ctx->last_K, nP = K * (K + 1) / 2, W = nP + K + 2;
  hipStream_t st = ctx->stream;
  const double *d_fx = (const double *)ctx->fxscal.p, *d_xm = d_fx + kMaxK;
  CodeCols cr{kColLsqR, (const double *)ctx->ffvecs.p, M, M};
  cr.fancy = (const double *)ctx->fancy.p;
  cr.xmean = d_xm;
  cr.ignore = (const uint8_t *)ctx->ignore_dev.p;
  cr.fxscal = d_fx;
  cr.K = K;
  CodeCols cg = cr;
  cg.kind = kColLsqG;
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const int64_t nblk_all = (M + 127) / 128;
  int64_t nr = (nind + 255) / 256 * 256, nb = std::min(nblk_all, kLsqRange);
  int32_t smax = 32;
  // with every individual selected, the selection's grouped codes are the individuals'
  const bool shared = ctx->sel_all && ctx->have_selg;
  const int64_t Gall = (M + kGrp - 1) / kGrp;
  CodesPlan pr, pg;
  size_t codes = 0;
  for (;;) {
    pr = eig_codes_plan(ctx->num_cu, kCdSum, K + 1, std::min<int64_t>(nr, nind), nb, smax);
    pg = eig_codes_plan(ctx->num_cu, kCdMiss, nP, std::min<int64_t>(nr, nind), nb, smax);
    codes = shared ? 0 : up((size_t)nr * nb * 32);
    const size_t need = pr.head_bytes + pg.head_bytes + up(pr.dig_bytes) + up(pg.dig_bytes) +
                        up(pr.part_bytes) + up(pg.part_bytes) + codes;
    if (need <= bytes) break;
    if (nb > 512) nb = (nb + 1) / 2;
    else if (smax > 4) smax /= 2;
    else if (nb > 64) nb = (nb + 1) / 2;
    else if (smax > 1) smax /= 2;
    else if (nr > 256) nr = std::max<int64_t>(256, nr / 2 / 256 * 256);
    else return eig_set_err(ctx, EIG_E_NOMEM, "lsqproject: workspace too small");
  }
  char *p = ws;
  auto take = [&](size_t b) {
    char *q = p;
    p += up(b);
    return q;
  };
  void *hr = take(pr.head_bytes), *hg = take(pg.head_bytes);
  void *dr = take(pr.dig_bytes), *dg = take(pg.dig_bytes);
  void *sr = take(pr.part_bytes), *sg = take(pg.part_bytes);
  uint4 *cd = (uint4 *)take(codes);
  EIG_TRY(eig_codes_scales(ctx, pr, cr, hr, st));
  EIG_TRY(eig_codes_scales(ctx, pg, cg, hg, st));
  for (int64_t q0 = 0; q0 < nind; q0 += nr) {
    const int64_t rows = std::min<int64_t>(nr, nind - q0), tiles = (rows + 127) / 128;
    for (int64_t s0 = 0; s0 < nblk_all; s0 += kLsqRange) {
      EIG_TRY(eig_codes_restart(ctx, pr, hr, st));
      EIG_TRY(eig_codes_restart(ctx, pg, hg, st));
      const int64_t s1 = std::min(nblk_all, s0 + kLsqRange);
      // a last, shorter chunk keeps the plan: SNPs past s1 have no digits
      cr.n = cg.n = std::min(M, s1 * 128);
      for (int64_t b0 = s0; b0 < s1; b0 += nb) {
        const int64_t G64 = 2 * nb;
        CodeView v{(const uint8_t *)cd, nullptr, G64 * 2048, 16, 4096, 2048, tiles * 128, G64 * 4,
                   kCodeGrouped};
        if (shared) {
          v.base = (const uint8_t *)ctx->selg.p + ((q0 >> 7) * Gall + 2 * b0) * 2048;
          v.RT = Gall * 2048;
          v.nword = (Gall - 2 * b0) * 4;
        } else {
          hipLaunchKernelGGL(k_regroup_geno, dim3((unsigned)((tiles * G64 + 1) / 2)), dim3(256), 0, st,
                             (const uint8_t *)ctx->geno.p, ctx->rlen, M, nind, b0 * 128, (int32_t)q0,
                             G64, tiles * G64, cd);
        }
        EIG_TRY(eig_codes_mul(ctx, pr, v, cr, b0, hr, dr, sr, b0 > s0, st));
        EIG_TRY(eig_codes_mul(ctx, pg, v, cg, b0, hg, dg, sg, b0 > s0, st));
      }
      double *a = acc + q0 * W;
      EIG_TRY(eig_codes_out_sum(ctx, pg, rows, hg, sg, 1.0, a, W, 1, nP, s0 > 0, st));
      EIG_TRY(eig_codes_out_sum(ctx, pr, rows, hr, sr, 1.0, a + nP, W, 1, K + 1, s0 > 0, st));
    }
  }
  return EIG_OK;
}

static int lsqproject(eig_ctx *ctx, const int32_t *use, const int32_t *itype, int32_t npop,
                      double *acoeffs, double *bcoeffs, int32_t *status) {
  if (!ctx || !use) return eig_set_err(ctx, EIG_E_ARG, "eig_lsqproject: args");
  if (!ctx->have_load) return eig_set_err(ctx, EIG_E_STATE, "eig_lsqproject before eig_loadings");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  const int64_t M = ctx->nsnp;
  const int32_t nind = ctx->nind, K = ctx->last_K;
  hipStream_t st = ctx->stream;
  const int nP = K * (K + 1) / 2, W = nP + K + 2;
  double *d_fill = nullptr;
  const int32_t *d_itype = nullptr;
  if (itype) EIG_TRY(eig_lsq_filltab(ctx, use, itype, npop, K, &d_fill, &d_itype));
  size_t out_b = 8 * (size_t)2 * K * nind + 4 * (size_t)nind * 2 + 256;
  EIG_TRY(eig_ensure(ctx, ctx->proj_out, out_b));
  double *d_ans = (double *)ctx->proj_out.p, *d_rhs = d_ans + (size_t)K * nind;
  int32_t *d_st = (int32_t *)(d_rhs + (size_t)K * nind), *d_use = d_st + nind;
  EIG_HIP(ctx, hipMemcpyAsync(d_use, use, 4 * (size_t)nind, hipMemcpyHostToDevice, st));
  EIG_HIP(ctx, hipMemsetAsync(d_ans, 0, 8 * (size_t)K * nind, st));
  const double *d_fx = (const double *)ctx->fxscal.p, *d_xm = d_fx + kMaxK;
  int64_t nchunk = 1;
  if (!itype) {
    // the normal equations from the code planes (5,000 x 600,000, K = 10: 2.3 against
    // 25.6 ms of FP64 sums per individual); the workspace holds up to 1 GiB of it at once
    const size_t acc_b = (8 * (size_t)nind * W + 255) & ~(size_t)255;
    const size_t work = std::min((size_t)1 << 30, ((size_t)nind + 4096) * (M + 4096) + ((size_t)64 << 20));
    EIG_TRY(eig_ensure(ctx, ctx->scratch2, acc_b + work));
    eig_time_begin(ctx);
    EIG_TRY(lsq_normal(ctx, (double *)ctx->scratch2.p, (char *)ctx->scratch2.p + acc_b, work));
  } else {
    // a fill's genotypes are FP64 values of their own: sums per individual
    nchunk = (M + kLsqChunk - 1) / kLsqChunk;
    const int32_t nblk = (nind + 63) / 64;
    EIG_TRY(eig_ensure(ctx, ctx->scratch2, 8 * (size_t)nchunk * nind * W));
    eig_time_begin(ctx);
    EIG_KSWITCH(K, hipLaunchKernelGGL((k_lsq_gram<KC>), dim3((unsigned)(nchunk * nblk)), dim3(64),
                                      0, st, (const uint8_t *)ctx->geno.p, ctx->rlen, M, nind,
                                      (const double *)ctx->ffvecs.p, d_fx,
                                      (const double *)ctx->fancy.p, d_xm,
                                      (const uint8_t *)ctx->ignore_dev.p, (const double *)d_fill,
                                      d_itype, npop, (double *)ctx->scratch2.p, nblk));
  }
  EIG_KSWITCH(K, hipLaunchKernelGGL((k_lsq_solve<KC>), dim3((unsigned)((nind + 63) / 64)), dim3(64), 0,
                                    st, (const double *)ctx->scratch2.p, nchunk, nind,
                                    (const int32_t *)d_use, d_itype, d_ans, d_rhs, d_st));
  EIG_HIP(ctx, hipGetLastError());
  eig_time_end(ctx, "lsqproject");
  std::vector<double> ans((size_t)K * nind), rhs((size_t)K * nind);
  std::vector<int32_t> sv(nind);
  EigFetch f(ctx);
  EIG_TRY(f.get(ans.data(), d_ans, 8 * (size_t)K * nind));
  EIG_TRY(f.get(rhs.data(), d_rhs, 8 * (size_t)K * nind));
  EIG_TRY(f.get(sv.data(), d_st, 4 * (size_t)nind));
  EIG_TRY(f.wait());
  // regans persists across individuals in the reference (smartpca.c:4656,
  // regsubs.c:51-53): a failed solve keeps the previous individual's answer.
  double last[kMaxK];
  for (int j = 0; j < K; ++j) last[j] = 0.0;
  for (int32_t q = 0; q < nind; ++q) {
    if (status) status[q] = sv[q];
    if (sv[q] == 0)
      for (int j = 0; j < K; ++j) last[j] = ans[(size_t)j * nind + q];
    if (sv[q] == 0 || sv[q] == 2)
      for (int j = 0; j < K; ++j)
        if (acoeffs) acoeffs[(size_t)j * nind + q] = last[j];
    if (bcoeffs && (sv[q] == 0 || sv[q] == 2))
      for (int j = 0; j < K; ++j) bcoeffs[(size_t)j * nind + q] = rhs[(size_t)j * nind + q];
  }
  return EIG_OK;
}

extern "C" int eig_lsqproject(eig_ctx *ctx, const int32_t *use, double *acoeffs,
                              double *bcoeffs, int32_t *status) {
  return lsqproject(ctx, use, nullptr, 0, acoeffs, bcoeffs, status);
}

extern "C" int eig_lsqproject_fill(eig_ctx *ctx, const int32_t *use, const int32_t *itype,
                                   int32_t npop, double *acoeffs, double *bcoeffs,
                                   int32_t *status) {
  if (!itype) return eig_set_err(ctx, EIG_E_ARG, "eig_lsqproject_fill: itype is required");
  return lsqproject(ctx, use, itype, npop, acoeffs, bcoeffs, status);
}

// ---------------------------------------------------------------- allocation-free lsqproject
namespace {
__global__ void k_lsq_clear(double *__restrict__ p, int64_t n) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e < n) p[e] = 0.0;
}

// the stale-answer rule of the reference, in individual order, one thread per axis j:
// outputs of individuals with status 1 or 3 keep the caller's values
__global__ void k_lsq_stale(const double *__restrict__ ans, const double *__restrict__ rhs,
                            const int32_t *__restrict__ st, int32_t nind, int32_t K,
                            double *__restrict__ A, double *__restrict__ B) {
  const int j = threadIdx.x;
  if (j >= K) return;
  double last = 0.0;
  for (int32_t q = 0; q < nind; ++q) {
    const int32_t s = st[q];
    if (s == 0) last = ans[(int64_t)j * nind + q];
    if (s == 0 || s == 2) {
      if (A) A[(int64_t)j * nind + q] = last;
      if (B) B[(int64_t)j * nind + q] = rhs[(int64_t)j * nind + q];
    }
  }
}
}  // namespace

extern "C" int eig_lsqproject_noalloc(eig_ctx *ctx, const int32_t *use, double *acoeffs,
                                      double *bcoeffs, int32_t *status) {
  if (!ctx || !use) return eig_set_err(ctx, EIG_E_ARG, "eig_lsqproject_noalloc: args");
  if (!ctx->have_load)
    return eig_set_err(ctx, EIG_E_STATE, "eig_lsqproject_noalloc before eig_loadings");
  if (!ctx->noalloc) return eig_set_err(ctx, EIG_E_STATE, "eig_lsqproject_noalloc: no workspace");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  const int32_t nind = ctx->nind, K = ctx->last_K;
  hipStream_t st = ctx->stream;
  const int nP = K * (K + 1) / 2, W = nP + K + 2;
  // workspace: acc | ans | rhs | A | B | status | use | the products' work area (at least the
  // size of acc, which holds chunks of it at every K)
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t per = (size_t)nind * W;
  const size_t o_acc = 0, o_ans = up(8 * per), o_rhs = o_ans + up(8 * (size_t)K * nind),
               o_A = o_rhs + up(8 * (size_t)K * nind), o_B = o_A + up(8 * (size_t)K * nind),
               o_st = o_B + up(8 * (size_t)K * nind), o_use = o_st + up(4 * (size_t)nind),
               o_part = o_use + up(4 * (size_t)nind);
  if (o_part + 8 * per > ctx->noalloc_bytes)
    return eig_set_err(ctx, EIG_E_ARG,
                       "eig_lsqproject_noalloc: %d individuals x K=%d need more than the %zu-byte "
                       "static workspace", nind, K, ctx->noalloc_bytes);
  char *base = (char *)ctx->noalloc;
  double *d_acc = (double *)(base + o_acc), *d_ans = (double *)(base + o_ans),
         *d_rhs = (double *)(base + o_rhs), *d_A = (double *)(base + o_A),
         *d_B = (double *)(base + o_B);
  int32_t *d_st = (int32_t *)(base + o_st), *d_use = (int32_t *)(base + o_use);
  const size_t kn = (size_t)K * nind;
  EIG_HIP(ctx, hipMemcpyAsync(d_use, use, 4 * (size_t)nind, hipMemcpyHostToDevice, st));
  // the caller's current outputs go in, so entries the rule leaves alone come back as they were
  if (acoeffs) EIG_HIP(ctx, hipMemcpyAsync(d_A, acoeffs, 8 * kn, hipMemcpyHostToDevice, st));
  if (bcoeffs) EIG_HIP(ctx, hipMemcpyAsync(d_B, bcoeffs, 8 * kn, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_lsq_clear, dim3((unsigned)((kn + 255) / 256)), dim3(256), 0, st, d_ans,
                     (int64_t)kn);
  EIG_TRY(lsq_normal(ctx, d_acc, base + o_part, ctx->noalloc_bytes - o_part));
  EIG_KSWITCH(K, hipLaunchKernelGGL((k_lsq_solve<KC>), dim3((unsigned)((nind + 63) / 64)), dim3(64), 0,
                                    st, (const double *)d_acc, (int64_t)1, nind,
                                    (const int32_t *)d_use, (const int32_t *)nullptr, d_ans, d_rhs,
                                    d_st));
  hipLaunchKernelGGL(k_lsq_stale, dim3(1), dim3(64), 0, st, (const double *)d_ans,
                     (const double *)d_rhs, (const int32_t *)d_st, nind, K, acoeffs ? d_A : nullptr,
                     bcoeffs ? d_B : nullptr);
  EIG_HIP(ctx, hipGetLastError());
  if (status) EIG_HIP(ctx, hipMemcpyAsync(status, d_st, 4 * (size_t)nind, hipMemcpyDeviceToHost, st));
  if (acoeffs) EIG_HIP(ctx, hipMemcpyAsync(acoeffs, d_A, 8 * kn, hipMemcpyDeviceToHost, st));
  if (bcoeffs) EIG_HIP(ctx, hipMemcpyAsync(bcoeffs, d_B, 8 * kn, hipMemcpyDeviceToHost, st));
  EIG_HIP(ctx, hipStreamSynchronize(st));
  return EIG_OK;
}
