// fastmode: randomized block-Krylov PCA of the normalised genotype matrix
// (kjg_fpca, ksrc/kjg_fpca.c:24-101, with setgval's normalisation, gval.c:31-87).
//
// X is the ncols x nrows matrix of SNP rows, X[m][i] = ((g - mean) * fancy) / sqrt(2)
// with mean = xmean / xfancy exactly as setgval recomputes it, and 0 for a missing
// genotype.  Omega (nrows x L) is a Gaussian panel; for i < I
//     Q_i = X Omega_i,   Omega_{i+1} = X^T Q_i / ncols,
// Q_I = X Omega_I; the columns of Q = [Q_0 .. Q_I] are orthonormalised (the
// reference takes the SVD of Q; here block Gram-Schmidt with reorthogonalisation,
// each block orthonormalised by Gram + Jacobi eigendecomposition, gives an
// orthonormal basis U of the same range); then B = X^T U, and the top-K left
// singular vectors of B (from the eigen-decomposition of B^T B) are the
// eigenvectors, S^2 / ncols the eigenvalues (kjg_fpca.c:79-95).
//
// The two panel products read X straight from packed codes: in the FP64 form as exact
// integer products with fixed-point digits of the panel (codes.hip), in the split-BF16
// form on BF16 MFMA (32x32x16) over hi/lo splits, each stage's operands loaded while the
// previous stage's MFMAs run (two LDS buffers, one barrier per stage).  The tall-skinny Gram and basis products run on the library's FP64
// MFMA GEMM (gemm.hip).

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "eig_internal.h"

namespace {
constexpr int kMaxCT = 16;    // column tiles of 16 -> at most 256 columns
constexpr int kJacMax = 256;  // order limit of the one-block Jacobi eigensolver
}  // namespace

// ---------------------------------------------------------------- levels
// lf[m][g] for g = 0,1,2 and lf[m][3] = 0 (missing); SNPs not live or with no
// observed genotype get zero rows.  Built without contraction (gval.c:73-80).
__global__ void k_fpca_levels(const double *__restrict__ mean, const double *__restrict__ fancy,
                              const int32_t *__restrict__ status, int64_t M,
                              double *__restrict__ lf) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  double *o = lf + 4 * m;
  const int32_t st = status[m];
  if (st == EIG_SNP_DEAD || st == EIG_SNP_ALLMISS) {
    o[0] = o[1] = o[2] = o[3] = 0.0;
    return;
  }
  const double f = fancy[m];
  const double xm = mean[m] * f;  // xmean[col] = pmean * yfancy (smartpca.c:3205)
  const double mu = xm / f;       // mean = xmean[col] / xfancy[col] (gval.c:74)
  const double r2 = sqrt(2.0);
  for (int k = 0; k < 3; ++k) {
    double y = (double)k - mu;
    y *= f;
    o[k] = y / r2;
  }
  o[3] = 0.0;
}

// ---------------------------------------------------------------- Gaussian panel
__device__ __host__ inline uint64_t fp_mix64(uint64_t x) {
  x ^= x >> 30;
  x *= 0xBF58476D1CE4E5B9ull;
  x ^= x >> 27;
  x *= 0x94D049BB133111EBull;
  x ^= x >> 31;
  return x;
}

// Omega[i][c] ~ N(0,1) for i < n, c < L (Box-Muller on a counter hash); zero padding.
__global__ void k_fpca_gauss(double *__restrict__ A, int32_t npad, int32_t lda, int32_t n,
                             int32_t L, uint64_t seed) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)npad * lda) return;
  const int32_t i = (int32_t)(idx / lda), c = (int32_t)(idx % lda);
  double z = 0.0;
  if (i < n && c < L) {
    const uint64_t key = (uint64_t)i * (uint64_t)L + (uint64_t)c;
    const uint64_t h1 = fp_mix64(seed + (key + 1) * 0x9E3779B97F4A7C15ull);
    const uint64_t h2 = fp_mix64(h1 ^ 0xD1B54A32D192ED03ull);
    const double u1 = ((double)(h1 >> 11) + 1.0) * 0x1.0p-53;  // (0, 1]
    const double u2 = (double)(h2 >> 11) * 0x1.0p-53;          // [0, 1)
    z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
  }
  A[idx] = z;
}

// out[i][c] = scale * sum_s part[s][i][c] (splits in order) for c < min(ldp, ldo);
// padding columns of out beyond ldp are left alone.
__global__ void k_fpca_reduce(const double *__restrict__ part, int32_t S, int64_t npad,
                              int32_t ldp, double scale, double *__restrict__ out, int32_t ldo) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= npad * ldp) return;
  const int64_t i = idx / ldp;
  const int c = (int)(idx % ldp);
  if (c >= ldo) return;
  double s = 0.0;
  for (int32_t k = 0; k < S; ++k) s += part[(int64_t)k * npad * ldp + idx];
  out[i * ldo + c] = scale * s;
}

// ---------------------------------------------------------------- split-BF16 panels
// The chosen form of the panel products: every operand is split into bf16 hi + lo
// and the four products hi*hi, hi*lo, lo*hi, lo*lo run on v_mfma_f32_32x32x16_bf16,
// in FP32 within a block of the reduction and promoted to FP64 across blocks (as
// the split-BF16 XTX).  The genotype operand is decoded straight into MFMA operand
// registers; the dense panel is split once per product into hi / lo MFMA operands.
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float fp_f32x16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 fp_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t fp_u32x4;

// fastmode levels lf as bf16 hi (low half) | lo (high half) per (SNP, code)
__global__ void k_fpca_levbf(const double *__restrict__ lf, int64_t M, uint32_t *__restrict__ lb) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 4 * M) return;
  const double v = lf[e];
  const uint16_t hi = eig_bf16_rne((float)v);
  const uint16_t lo = eig_bf16_rne((float)(v - (double)eig_bf16_to_f32(hi)));
  lb[e] = (uint32_t)hi | ((uint32_t)lo << 16);
}

// The dense panel src[k * lds + c] (k < rows, c < C; zero past them) as bf16 hi / lo MFMA
// operands: column group cg of 32 CT columns, 16-row step s, 32-column tile ct and part hl
// (0 hi, 1 lo) fill 1 KB at frag + (((cg nstep + s) CT + ct) 2 + hl) * 512, lane l's eight
// values at 8 l: column l % 32, rows 8 (l / 32) + 0 .. 7.  A stage of the products is one
// contiguous piece, staged and read without padding or bank conflicts.
__global__ __launch_bounds__(256) void k_fpca_split(const double *__restrict__ src, int64_t rows,
                                                    int64_t lds, int32_t C, int64_t nstep,
                                                    int32_t CT, uint16_t *__restrict__ frag) {
  __shared__ double tile[32][33];
  const int64_t r0 = (int64_t)blockIdx.x * 32;
  const int32_t c0 = blockIdx.y * 32;
  const int t = threadIdx.x, tx = t & 31, ty = t >> 5;  // 8 rows at a time
  for (int k = ty; k < 32; k += 8) {
    const int64_t r = r0 + k;
    const int32_t c = c0 + tx;
    tile[k][tx] = (r < rows && c < C) ? src[r * lds + c] : 0.0;
  }
  __syncthreads();
  const int s = t >> 7, hl = (t >> 6) & 1, lane = t & 63, h = lane >> 5;
  const int64_t step = 2 * (int64_t)blockIdx.x + s;
  if (step >= nstep) return;
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const double v = tile[16 * s + 8 * h + j][lane & 31];
    const uint16_t hi = eig_bf16_rne((float)v);
    const uint16_t lo = eig_bf16_rne((float)(v - (double)eig_bf16_to_f32(hi)));
    const uint32_t x = hl ? lo : hi;
    o[j >> 1] = (j & 1) ? o[j >> 1] | (x << 16) : x;
  }
  const int32_t cg = blockIdx.y / CT, ct = blockIdx.y % CT;
  *(uint4 *)(frag + ((((int64_t)cg * nstep + step) * CT + ct) * 2 + hl) * 512 + lane * 8) =
      make_uint4(o[0], o[1], o[2], o[3]);
}

// Y = X A.  Persistent over SNP tiles of 128 (4 waves x 32 SNPs); a wave's 32 SNPs x 32 CT
// columns accumulate in FP32 over blkt sample tiles, then in FP64.  A lane of the genotype
// operand is one SNP for the whole sum, so its four levels stay in registers and two codes
// become an operand word by one v_perm_b32 each for hi and lo, with a selector both share:
// no table, and LDS (128 bytes a cycle) carries the panel alone.  A table of level pairs in
// LDS took eight lookups a step, as many LDS cycles as the step has MFMA cycles: at 100,000
// x 500,000 and 20 columns 12.9 ms, now 11.0 (1.16 PFLOP/s; the matrix units are busy 61 % of
// the cycles at the 1.8 GHz this load leaves, the decode's 26 VALU instructions a step the
// rest).  Panel
// stages of half a sample tile (four steps), global -> registers -> one of two LDS buffers,
// one barrier per stage.
template <int CT>
__global__ __launch_bounds__(256, CT == 1 ? 4 : 2) void k_fpca_xa_bf16(
    const uint32_t *__restrict__ sel, int64_t M, int32_t nst, const uint32_t *__restrict__ lbf,
    const uint16_t *__restrict__ frag, double *__restrict__ Y, int64_t ldy, int32_t C, int32_t blkt) {
  constexpr int kPan = 512 * CT;  // 16-byte pieces of a stage's panel
  __shared__ fp_u32x4 sA[2][kPan];
  const int t = threadIdx.x, w = t >> 6, lane = t & 63, h = lane >> 5, r = lane & 31;
  const int64_t ntiles = (M + 127) / 128;
  const int32_t nstage = 2 * nst;
  // rotations that bring the lane's eight codes down (codes 0, 2, 4, 6 at bits 0, 4, 8, 12)
  // and the odd ones to bits 16, 20, 24, 28
  const uint32_t rot0 = 16u * (uint32_t)h, rot1 = (18u + 16u * (uint32_t)h) & 31u;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t mb = tile * 128, m = mb + 32 * w + r;  // this lane's SNP
    const int64_t mr = m < M ? m : M - 1;  // one past M reads SNP M-1's words, its levels are 0
    fp_u32x4 lv = *(const fp_u32x4 *)(lbf + 4 * mr);
    if (m >= M) lv = fp_u32x4{0u, 0u, 0u, 0u};
    const uint32_t h01 = (lv[0] & 0xFFFFu) | (lv[1] << 16), h23 = (lv[2] & 0xFFFFu) | (lv[3] << 16);
    const uint32_t l01 = (lv[0] >> 16) | (lv[1] & 0xFFFF0000u), l23 = (lv[2] >> 16) | (lv[3] & 0xFFFF0000u);
    fp_u32x4 pa[2 * CT], wd;
    auto fetch = [&](int32_t g) {
      const fp_u32x4 *p = (const fp_u32x4 *)frag + (int64_t)g * kPan + t;
#pragma unroll
      for (int j = 0; j < 2 * CT; ++j) pa[j] = p[256 * j];
      wd = *((const fp_u32x4 *)(sel + ((int64_t)(g >> 1) * M + mr) * kTileWords) + (g & 1));
    };
    fp_f32x16 acc[CT];
    double dacc[CT][16];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        acc[ct][q] = 0.f;
        dacc[ct][q] = 0.0;
      }
    auto promote = [&]() {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          dacc[ct][q] += (double)acc[ct][q];
          acc[ct][q] = 0.f;
        }
    };
    fetch(0);
    __syncthreads();  // the previous tile's panel reads are done
    int32_t left = 2 * blkt;
    int buf = 0;
    for (int32_t g = 0; g < nstage; ++g) {
#pragma unroll
      for (int j = 0; j < 2 * CT; ++j) sA[buf][t + 256 * j] = pa[j];
      const fp_u32x4 cw = wd;  // this stage's words; wd takes the next stage's
      // the other buffer was last read before this barrier's previous instance
      __syncthreads();
      if (g + 1 < nstage) fetch(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t x = cw[j];
        // bytes: codes 0 | 2 << 4, 4 | 6 << 4, 1 | 3 << 4, 5 | 7 << 4 (and other bits)
        const uint32_t p = (__builtin_amdgcn_alignbit(x, x, rot0) & 0xFFFFu) |
                           (__builtin_amdgcn_alignbit(x, x, rot1) & 0xFFFF0000u);
        // byte selectors 2 c and 2 c + 1 of codes 0, 4, 1, 5, then of 2, 6, 3, 7
        const uint32_t a0 = (p << 1) & 0x06060606u, a1 = a0 | 0x01010101u;
        const uint32_t b0 = (p >> 3) & 0x06060606u, b1 = b0 | 0x01010101u;
        const uint32_t sl[4] = {__builtin_amdgcn_perm(a1, a0, 0x06020400u),
                                __builtin_amdgcn_perm(b1, b0, 0x06020400u),
                                __builtin_amdgcn_perm(a1, a0, 0x07030501u),
                                __builtin_amdgcn_perm(b1, b0, 0x07030501u)};
        fp_u32x4 xh, xl;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          xh[q] = __builtin_amdgcn_perm(h23, h01, sl[q]);
          xl[q] = __builtin_amdgcn_perm(l23, l01, sl[q]);
        }
        const fp_bf16x8 ah = __builtin_bit_cast(fp_bf16x8, xh), al = __builtin_bit_cast(fp_bf16x8, xl);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const fp_bf16x8 bh = __builtin_bit_cast(fp_bf16x8, sA[buf][(j * CT + ct) * 128 + lane]);
          const fp_bf16x8 bl = __builtin_bit_cast(fp_bf16x8, sA[buf][(j * CT + ct) * 128 + 64 + lane]);
          acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bl, acc[ct], 0, 0, 0);
          acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc[ct], 0, 0, 0);
          acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc[ct], 0, 0, 0);
          acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc[ct], 0, 0, 0);
        }
      }
      if (--left == 0) {
        promote();
        left = 2 * blkt;
      }
      buf ^= 1;
    }
    promote();
    // accumulator: lane l, element q -> row 8(q>>2) + 4(l>>5) + (q&3), column l&31
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int64_t row = mb + 32 * w + 8 * (q >> 2) + 4 * h + (q & 3);
        const int col = 32 * ct + r;
        if (row < M && col < C) Y[row * ldy + col] = dacc[ct][q];
      }
  }
}

// Level tables of X^T B: per 64-SNP group 512 words of hi pairs, then 512 of lo pairs.  Word
// ((s4 4 + q) 2 + h) 16 + c holds the levels of SNPs 16 s4 + 2 (4 h + q) + {0, 1} for codes
// c & 3 and c >> 2, one dword of the operand (the split-BF16 XTX's scheme); zero past M.
constexpr int kFpTab = 4 * 4 * 2 * 16;
__global__ __launch_bounds__(256) void k_fpca_tab(const uint32_t *__restrict__ lbf, int64_t M, int64_t G64,
                                                  uint32_t *__restrict__ tab) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t g = i / kFpTab;
  if (g >= G64) return;
  const int e = (int)(i % kFpTab);
  const int s4 = e >> 7, q = (e >> 5) & 3, hh = (e >> 4) & 1, c = e & 15;
  const int64_t m = g * kGrp + 16 * s4 + 2 * (4 * hh + q);
  const uint32_t e0 = m < M ? lbf[4 * m + (c & 3)] : 0u;
  const uint32_t e1 = m + 1 < M ? lbf[4 * (m + 1) + (c >> 2)] : 0u;
  tab[2 * kFpTab * g + e] = (e0 & 0xFFFFu) | (e1 << 16);
  tab[2 * kFpTab * g + kFpTab + e] = (e0 >> 16) | (e1 & 0xFFFF0000u);
}

// Partial X^T B.  One block per item (sample tile, SNP split, column group of 32 NCT): one
// sample tile (4 waves x 32 samples) x 32 NCT columns over SNPs [s*mchunk, ...) (mchunk a
// multiple of 64).  The genotype operand comes from the grouped layout by lookups in the
// group's level table, the panel operand from frag (k_fpca_split's layout); table and panel
// stage of a group go global -> registers -> one of two LDS buffers as they lie in memory,
// one barrier per group: no address arithmetic or packing in the loop, five waves per SIMD
// (32 columns) and three (64) instead of three and two.  At 100,000 x 500,000 12.3 -> 10.0 ms
// with 20 columns, 62.7 -> 52.4 with 192 (1.47 PFLOP/s, the matrix units busy 69 % of the
// cycles at 2 GHz).  part[s][i][c] with row stride ldp.
template <int NCT>
__global__ __launch_bounds__(256, NCT == 1 ? 4 : 2) void k_fpca_xtb_bf16(
    const uint2 *__restrict__ selg, int64_t G64, int64_t M, int32_t nst,
    const uint32_t *__restrict__ tabs, const uint16_t *__restrict__ frag, int32_t S, int64_t mchunk,
    int32_t blkg, double *__restrict__ part, int32_t ldp) {
  constexpr int GW = 32 * NCT;          // columns per group
  constexpr int kPan = 512 * NCT;       // 16-byte pieces of a group's panel
  constexpr int kLo = kFpTab / 4 + 1;   // the lo table starts 2064 bytes on: no paired LDS load spans it
  __shared__ fp_u32x4 sT[2][2 * kFpTab / 4 + 1], sB[2][kPan];
  const int t = threadIdx.x, w = t >> 6, lane = t & 63, h = lane >> 5, r = lane & 31;
  const int64_t npad = (int64_t)nst * kTileS;
  const int64_t it = blockIdx.x;
  const int32_t st = (int32_t)(it % nst);
  const int64_t rest = it / nst;
  const int32_t s = (int32_t)(rest % S), cg = (int32_t)(rest / S);
  const int64_t m_begin = (int64_t)s * mchunk;
  const int64_t m_end = min(M, m_begin + mchunk);
  double *out = part + ((int64_t)s * npad + (int64_t)st * kTileS) * ldp;
  if (m_begin >= m_end) {  // an empty split (M not filling S chunks): zero partial
    for (int e = t; e < kTileS * GW; e += 256) out[(int64_t)(e / GW) * ldp + GW * cg + e % GW] = 0.0;
    return;
  }
  const int32_t ng = (int32_t)((m_end - m_begin + kGrp - 1) / kGrp);
  const int64_t g0 = m_begin / kGrp;
  const uint2 *src = selg + (((int64_t)st * G64 + g0) * kTileS + 32 * w + r) * 2 + h;
  const fp_u32x4 *tsrc = (const fp_u32x4 *)tabs + g0 * 256 + t;
  const fp_u32x4 *psrc = (const fp_u32x4 *)frag + ((int64_t)cg * G64 + g0) * kPan + t;
  const int tdst = t < 128 ? t : t + 1;
  fp_u32x4 tv, pv[2 * NCT];
  auto fetch = [&]() {
    tv = *tsrc;
#pragma unroll
    for (int u = 0; u < 2 * NCT; ++u) pv[u] = psrc[256 * u];
  };
  auto store = [&](int buf) {
    sT[buf][tdst] = tv;
#pragma unroll
    for (int u = 0; u < 2 * NCT; ++u) sB[buf][t + 256 * u] = pv[u];
  };
  fp_f32x16 acc[NCT];
  double dacc[NCT][16];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      acc[ct][q] = 0.f;
      dacc[ct][q] = 0.0;
    }
  auto promote = [&]() {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        dacc[ct][q] += (double)acc[ct][q];
        acc[ct][q] = 0.f;
      }
  };
  uint2 cur = src[0], nxt;
  fetch();
  store(0);
  __syncthreads();
  int32_t left = blkg;
  for (int32_t gi = 0; gi < ng; ++gi) {
    const int buf = gi & 1;
    if (gi + 1 < ng) {  // the last group loads itself again
      src += 2 * kTileS;
      tsrc += 256;
      psrc += kPan;
    }
    nxt = *src;
    fetch();
    const uint32_t *th = (const uint32_t *)&sT[buf][0] + 16 * h, *tl = (const uint32_t *)&sT[buf][kLo] + 16 * h;
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const uint32_t word = (s4 < 2) ? cur.x : cur.y;
      fp_u32x4 xh, xl;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t c = (word >> (16 * (s4 & 1) + 4 * q)) & 15u;
        xh[q] = th[(s4 * 4 + q) * 32 + c];
        xl[q] = tl[(s4 * 4 + q) * 32 + c];
      }
      const fp_bf16x8 ah = __builtin_bit_cast(fp_bf16x8, xh), al = __builtin_bit_cast(fp_bf16x8, xl);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const fp_bf16x8 bh = __builtin_bit_cast(fp_bf16x8, sB[buf][(s4 * NCT + ct) * 128 + lane]);
        const fp_bf16x8 bl = __builtin_bit_cast(fp_bf16x8, sB[buf][(s4 * NCT + ct) * 128 + 64 + lane]);
        acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bl, acc[ct], 0, 0, 0);
        acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc[ct], 0, 0, 0);
        acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc[ct], 0, 0, 0);
        acc[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc[ct], 0, 0, 0);
      }
    }
    if (--left == 0) {
      promote();
      left = blkg;
    }
    store(buf ^ 1);
    cur = nxt;
    __syncthreads();
  }
  promote();
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int row = 32 * w + 8 * (q >> 2) + 4 * h + (q & 3);
      out[(int64_t)row * ldp + GW * cg + 32 * ct + r] = dacc[ct][q];
    }
}

// ---------------------------------------------------------------- Jacobi
// All eigenpairs of a symmetric n x n matrix (n <= 256, column-major, lda) by
// cyclic two-sided Jacobi with round-robin pairing, in one block.  On exit the
// diagonal of A holds the eigenvalues and V (n x n, ldv) their eigenvectors in
// its columns (unsorted).  Stops after a sweep in which no pair had
// |a_pq| > tol * sqrt(|a_pp a_qq|), or after max_sweeps.
__global__ __launch_bounds__(1024) void k_jacobi(double *__restrict__ A, int32_t lda,
                                                 double *__restrict__ V, int32_t ldv, int32_t n,
                                                 int32_t max_sweeps, double tol,
                                                 int32_t *__restrict__ sweeps_out) {
  __shared__ int32_t idx[kJacMax];
  __shared__ int32_t pp[kJacMax / 2], pq[kJacMax / 2];
  __shared__ double cs[kJacMax / 2], sn[kJacMax / 2];
  __shared__ int rotated;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int np = n + (n & 1);  // an odd order gets a dummy index n
  const int half = np / 2;
  for (int e = tid; e < n * n; e += nt) {
    const int i = e % n, j = e / n;
    V[(int64_t)j * ldv + i] = (i == j) ? 1.0 : 0.0;
  }
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    if (tid == 0) rotated = 0;
    for (int e = tid; e < np; e += nt) idx[e] = e;
    __syncthreads();
    for (int round = 0; round < np - 1; ++round) {
      for (int k = tid; k < half; k += nt) {
        int p = idx[k], q = idx[np - 1 - k];
        if (p > q) {
          const int t = p;
          p = q;
          q = t;
        }
        double c = 1.0, s = 0.0;
        if (q < n) {
          const double apq = A[(int64_t)q * lda + p];
          const double app = A[(int64_t)p * lda + p], aqq = A[(int64_t)q * lda + q];
          if (fabs(apq) > tol * sqrt(fabs(app * aqq)) && apq != 0.0) {
            const double tau = (aqq - app) / (2.0 * apq);
            const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
            c = 1.0 / sqrt(1.0 + t * t);
            s = t * c;
            rotated = 1;
          }
        }
        pp[k] = p;
        pq[k] = q < n ? q : p;
        cs[k] = c;
        sn[k] = q < n ? s : 0.0;
      }
      __syncthreads();
      // columns: A <- A J, V <- V J
      for (int e = tid; e < n * half; e += nt) {
        const int i = e % n, k = e / n;
        const double c = cs[k], s = sn[k];
        if (s == 0.0) continue;
        const int p = pp[k], q = pq[k];
        double *ap = A + (int64_t)p * lda + i, *aq = A + (int64_t)q * lda + i;
        const double x = *ap, y = *aq;
        *ap = c * x - s * y;
        *aq = s * x + c * y;
        double *vp = V + (int64_t)p * ldv + i, *vq = V + (int64_t)q * ldv + i;
        const double u = *vp, v = *vq;
        *vp = c * u - s * v;
        *vq = s * u + c * v;
      }
      __syncthreads();
      // rows: A <- J^T A
      for (int e = tid; e < n * half; e += nt) {
        const int j = e % n, k = e / n;
        const double c = cs[k], s = sn[k];
        if (s == 0.0) continue;
        const int p = pp[k], q = pq[k];
        double *ap = A + (int64_t)j * lda + p, *aq = A + (int64_t)j * lda + q;
        const double x = *ap, y = *aq;
        *ap = c * x - s * y;
        *aq = s * x + c * y;
      }
      __syncthreads();
      // exact zeros for the annihilated pairs
      for (int k = tid; k < half; k += nt)
        if (sn[k] != 0.0) {
          A[(int64_t)pq[k] * lda + pp[k]] = 0.0;
          A[(int64_t)pp[k] * lda + pq[k]] = 0.0;
        }
      // next pairing: keep idx[0], rotate idx[1..np-1] by one (np <= 256 < threads)
      {
        const int e = tid + 1;
        int v = 0;
        if (e < np) v = (e == 1) ? idx[np - 1] : idx[e - 1];
        __syncthreads();
        if (e < np) idx[e] = v;
        __syncthreads();
      }
    }
    if (!rotated) break;
    __syncthreads();
  }
  if (tid == 0) *sweeps_out = sweep;
}

// ---------------------------------------------------------------- host side
namespace {
struct Plan {
  int64_t M;
  int32_t nst, npad;
  const uint32_t *sel;
  const double *lf;
};
}  // namespace

// The orthonormalising factor of a block of n <= kJacLds columns from their Gram matrix G
// (column-major, ld n): with G = D S D (D the columns' norms) and S = Z diag(w) Z^T,
// w descending, the columns k of V = D^-1 Z diag(w)^-1/2 whose w_k > 1e-13 w_0; *keep their
// number (0 when S has no positive eigenvalue, -1 when the Jacobi sweeps ran out).  One
// block, everything in LDS: cyclic Jacobi in which a thread owns a 2 x 2 block of (row
// pair, column pair) and applies both rotations to it, two barriers a round (the
// column and row passes one by one took five more); the scaling, the order and the cut,
// with their copies and waits, were the host's (2.9 of the 18 ms that a basis of 11 x 20
// columns of 100,003 takes).
constexpr int kJacLds = 48;
__global__ __launch_bounds__(256) void k_orth_lds(const double *__restrict__ G, double *__restrict__ V,
                                                  int32_t n, int32_t max_sweeps, double tol,
                                                  int32_t *__restrict__ keep) {
  __shared__ double sA[kJacLds][kJacLds + 1], sV[kJacLds][kJacLds + 1], dsc[kJacLds];
  __shared__ double cs[kJacLds / 2], sn[kJacLds / 2];
  __shared__ int32_t pp[kJacLds / 2], pq[kJacLds / 2], rank[kJacLds];
  __shared__ int rotated, nkeep;
  const int tid = threadIdx.x;
  const int np = n + (n & 1);  // an odd order gets a dummy index n
  const int half = np / 2;
  if (tid < n) {
    const double g = G[(int64_t)tid * n + tid];
    dsc[tid] = g > 0.0 ? sqrt(g) : 1.0;
  }
  if (tid == 0) nkeep = 0;
  __syncthreads();
  for (int e = tid; e < n * n; e += 256) {  // sA[j][i] = column j, row i
    const int i = e % n, j = e / n;
    sA[j][i] = G[e] / (dsc[i] * dsc[j]);
    sV[j][i] = (i == j) ? 1.0 : 0.0;
  }
  __syncthreads();
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    if (tid == 0) rotated = 0;
    __syncthreads();
    for (int round = 0; round < np - 1; ++round) {
      if (tid < half) {
        // round robin: slot 0 holds index 0, slot s index 1 + (s - 1 - round) mod (np - 1)
        const int s0 = tid, s1 = np - 1 - tid;
        auto at = [&](int s) {
          const int v = s - 1 - round;
          return s == 0 ? 0 : 1 + (v < 0 ? v + np - 1 : v);
        };
        const int x = at(s0), y = at(s1);
        const int p = x < y ? x : y, q = x < y ? y : x;
        double c = 1.0, s = 0.0;
        if (q < n) {
          const double apq = sA[q][p], app = sA[p][p], aqq = sA[q][q];
          if (fabs(apq) > tol * sqrt(fabs(app * aqq)) && apq != 0.0) {
            const double tau = (aqq - app) / (2.0 * apq);
            const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
            c = 1.0 / sqrt(1.0 + t * t);
            s = t * c;
            rotated = 1;
          }
        }
        pp[tid] = p;
        pq[tid] = q;
        cs[tid] = c;
        sn[tid] = s;
      }
      __syncthreads();
      // A <- J^T A J, block (row pair k, column pair l)
      for (int l = tid >> 4; l < half; l += 16)
        for (int k = tid & 15; k < half; k += 16) {
          const double ck = cs[k], sk = sn[k], cl = cs[l], sl = sn[l];
          if (sk == 0.0 && sl == 0.0) continue;
          const int p = pp[k], q = pq[k], r = pp[l], u = pq[l];
          const bool hq = q < n, hu = u < n;
          const double a00 = sA[r][p], a10 = hq ? sA[r][q] : 0.0, a01 = hu ? sA[u][p] : 0.0,
                       a11 = hq && hu ? sA[u][q] : 0.0;
          // columns first: (r, u) <- (cl r - sl u, sl r + cl u), then rows likewise
          const double b00 = cl * a00 - sl * a01, b01 = sl * a00 + cl * a01;
          const double b10 = cl * a10 - sl * a11, b11 = sl * a10 + cl * a11;
          const bool diag = k == l && sk != 0.0;  // the annihilated pair: exact zeros
          sA[r][p] = ck * b00 - sk * b10;
          if (hu) sA[u][p] = diag ? 0.0 : ck * b01 - sk * b11;
          if (hq) sA[r][q] = diag ? 0.0 : sk * b00 + ck * b10;
          if (hq && hu) sA[u][q] = sk * b01 + ck * b11;
        }
      for (int k = tid >> 5; k < half; k += 8)  // V <- V J
        for (int i = tid & 31; i < n; i += 32) {
          const double c = cs[k], s = sn[k];
          if (s == 0.0) continue;
          const int p = pp[k], q = pq[k];
          const double u = sV[p][i], v = sV[q][i];
          sV[p][i] = c * u - s * v;
          sV[q][i] = s * u + c * v;
        }
      __syncthreads();
    }
    if (!rotated) break;
    __syncthreads();
  }
  // descending order, ties by index
  if (tid < n) {
    const double w = sA[tid][tid];
    double w0 = w;
    int r = 0;
    for (int j = 0; j < n; ++j) {
      const double x = sA[j][j];
      w0 = fmax(w0, x);
      r += x > w || (x == w && j < tid);
    }
    rank[tid] = r;
    if (w0 > 0.0 && w > 1e-13 * w0) atomicAdd(&nkeep, 1);
  }
  __syncthreads();
  for (int e = tid; e < n * n; e += 256) {
    const int i = e % n, j = e / n;
    V[(int64_t)rank[j] * n + i] = sV[j][i] / (sqrt(sA[j][j]) * dsc[i]);
  }
  if (tid == 0) *keep = sweep >= max_sweeps ? -1 : nkeep;
}

// V column k = work column ord[k] (n x n, column-major)
__global__ void k_gather_cols(double *__restrict__ V, const double *__restrict__ work,
                              const int32_t *__restrict__ ord, int32_t n) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)n * n) return;
  const int32_t k = (int32_t)(e / n), i = (int32_t)(e % n);
  V[e] = work[(int64_t)ord[k] * n + i];
}

// C (m x n, column-major, ld ldc) = sum over s of part[s] (m x n, ld m): 256 / T elements
// a block, T threads each summing every T-th part, then those sums in order
template <int T>
__global__ __launch_bounds__(256) void k_sum_parts(const double *__restrict__ part, int32_t S,
                                                   int32_t m, int32_t n, double *__restrict__ C,
                                                   int32_t ldc) {
  constexpr int E = 256 / T;
  __shared__ double sm[T][E];
  const int l = threadIdx.x % E, g = threadIdx.x / E;
  const int64_t e = (int64_t)blockIdx.x * E + l, mn = (int64_t)m * n;
  double v = 0.0;
  if (e < mn) {
#pragma unroll 8
    for (int32_t sp = g; sp < S; sp += T) v += part[(int64_t)sp * mn + e];
  }
  sm[g][l] = v;
  __syncthreads();
  if (g == 0 && e < mn) {
    for (int u = 1; u < T; ++u) v += sm[u][l];
    C[(e / m) * ldc + (e % m)] = v;
  }
}

// C_z (m x n, column-major, ld ldc, at C + z sC) = A_z B_z^T over chunk z's k (A and B
// column-major, sA and sB from chunk to chunk): k_gemm_f64's MFMAs in its order, element by
// element the same bits, but a wave per 16 x 16 tile instead of four per 64 x 64.  The sum
// over k is a serial chain of MFMAs (64 cycles each) that must not be cut, so skinny products
// take as many waves as they have tiles, each with its own loads, eight steps ahead.  All of
// them at 100,000 x 500,000 took 27 ms a call by k_gemm_f64, 12 now.
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double fp_f64x4;
__global__ __launch_bounds__(256) void k_gemm_nt_waves(int32_t m, int32_t n, int64_t k,
                                                       const double *__restrict__ A, int64_t lda, int64_t sA,
                                                       const double *__restrict__ B, int64_t ldb, int64_t sB,
                                                       double *__restrict__ C, int64_t ldc, int64_t sC) {
  constexpr int U = 8;
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int32_t mt = (m + 15) / 16, nt = (n + 15) / 16;
  const int32_t tile = (int32_t)blockIdx.x * 4 + (int32_t)(threadIdx.x >> 6);
  if (tile >= mt * nt) return;
  const int32_t i0 = (tile % mt) * 16, j0 = (tile / mt) * 16;
  // rows past the end read the last one and are not stored
  const double *pa = A + (int64_t)blockIdx.y * sA + min(i0 + r, m - 1) + q * lda;
  const double *pb = B + (int64_t)blockIdx.y * sB + min(j0 + r, n - 1) + q * ldb;
  auto ld = [&](int64_t s0, double (&a)[U], double (&b)[U]) {
    if (4 * (s0 + U) <= k) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        a[u] = pa[4 * (s0 + u) * lda];
        b[u] = pb[4 * (s0 + u) * ldb];
      }
    } else {  // zeros past k, which leave the sums as they are
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = 4 * (s0 + u) + q < k;
        a[u] = in ? pa[4 * (s0 + u) * lda] : 0.0;
        b[u] = in ? pb[4 * (s0 + u) * ldb] : 0.0;
      }
    }
  };
  fp_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  auto mma = [&](const double (&a)[U], const double (&b)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(b[u], a[u], acc, 0, 0, 0);
  };
  const int64_t steps = (k + 3) / 4;
  double a0[U], b0[U], a1[U], b1[U];
  ld(0, a0, b0);
  for (int64_t s = 0; s < steps; s += 2 * U) {
    ld(s + U, a1, b1);
    mma(a0, b0);
    ld(s + 2 * U, a0, b0);
    mma(a1, b1);
  }
  C += (int64_t)blockIdx.y * sC;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int32_t row = i0 + r, col = j0 + q + 4 * e;
    if (row < m && col < n) C[row + col * ldc] = acc[e];
  }
}

// C (m x n, column-major, ld ldc) = A B^T, A m x k (ld lda) and B n x k (ld ldb) column-major,
// for a long k: k is cut into S equal chunks (one batched product) and a remainder,
// whose partial products are summed.  A single product of these shapes has only a few
// output tiles to spread a long k over.  `fine`: chunks for 1,024 blocks, of at least 256 k
// (k = 100,003: 27 us a product against 140 in up to 64 chunks of at least 4,096, 24 to 96
// blocks).  The split-BF16 form keeps the coarse chunks and their order of summation: it
// rounds the basis to BF16 pairs, so a basis that differs in the last bits moves its
// eigenvectors by that form's own error over their gaps (1.6e-5 on a panel of twelve
// populations of like drift).
static int gemm_nt_long(eig_ctx *ctx, bool fine, int32_t m, int32_t n, int64_t k, const double *A,
                        int64_t lda, const double *B, int64_t ldb, double *C, int32_t ldc,
                        double *part, size_t part_doubles, hipStream_t st) {
  const int64_t mn = (int64_t)m * n;
  const int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 63) / 64);
  int64_t S = fine ? std::min<int64_t>(std::max<int64_t>(1, 1024 / tiles), k / 256)
                   : std::min<int64_t>(64, k / 4096);
  S = std::min<int64_t>(S, (int64_t)(part_doubles / std::max<int64_t>(mn, 1)) - 1);
  // skinny products of the coarse chunks: a wave per tile, the same bits
  auto mul = [&](int64_t kk, const double *a, int64_t sA, const double *b, int64_t sB, double *c, int64_t ldr,
                 int32_t batch) -> int {
    if (fine || n > 32)
      return eig_gemm_f64(ctx, st, false, true, m, n, kk, 1.0, a, lda, sA, b, ldb, sB, 0.0, c, ldr, mn, batch);
    const int32_t wv = ((m + 15) / 16) * ((n + 15) / 16);
    hipLaunchKernelGGL(k_gemm_nt_waves, dim3((unsigned)((wv + 3) / 4), (unsigned)batch), dim3(256), 0, st, m, n,
                       kk, a, lda, sA, b, ldb, sB, c, ldr, mn);
    EIG_HIP(ctx, hipGetLastError());
    return EIG_OK;
  };
  if (S < 2) return mul(k, A, 0, B, 0, C, ldc, 1);
  const int64_t kc = k / S, rem = k - S * kc;
  EIG_TRY(mul(kc, A, kc * lda, B, kc * ldb, part, m, (int32_t)S));
  int32_t nparts = (int32_t)S;
  if (rem > 0) {
    EIG_TRY(mul(rem, A + S * kc * lda, 0, B + S * kc * ldb, 0, part + S * mn, m, 1));
    ++nparts;
  }
  if (fine)
    hipLaunchKernelGGL(k_sum_parts<4>, dim3((unsigned)((mn + 63) / 64)), dim3(256), 0, st,
                       (const double *)part, nparts, m, n, C, ldc);
  else
    hipLaunchKernelGGL(k_sum_parts<1>, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, st,
                       (const double *)part, nparts, m, n, C, ldc);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

// Eigen-decomposition of the n x n symmetric device matrix G (column-major, ld n) of more
// than kJacLds columns: eigenvalues descending in w (host), eigenvectors in the columns of
// V (device, ld n) in the same order.
static int small_eigh(eig_ctx *ctx, double *G, int32_t n, double *V, std::vector<double> &w,
                      double *work, int32_t *d_sweeps) {
  if (n > kJacMax) return eig_set_err(ctx, EIG_E_ARG, "fpca: basis larger than %d", kJacMax);
  hipStream_t st = ctx->stream;
  hipLaunchKernelGGL(k_jacobi, dim3(1), dim3(1024), 0, st, G, n, work, n, n, 30, 1e-15, d_sweeps);
  EIG_HIP(ctx, hipGetLastError());
  std::vector<double> a((size_t)n * n);
  int32_t sweeps = 0;
  EIG_HIP(ctx, hipMemcpyAsync(a.data(), G, sizeof(double) * n * n, hipMemcpyDeviceToHost, st));
  EIG_HIP(ctx, hipMemcpyAsync(&sweeps, d_sweeps, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  EIG_HIP(ctx, hipStreamSynchronize(st));
  if (sweeps >= 30) return eig_set_err(ctx, EIG_E_CONVERGE, "fpca: Jacobi did not converge");
  std::vector<int32_t> ord(n);
  for (int32_t i = 0; i < n; ++i) ord[i] = i;
  std::stable_sort(ord.begin(), ord.end(), [&](int32_t x, int32_t y) {
    return a[(size_t)x * n + x] > a[(size_t)y * n + y];
  });
  w.resize(n);
  for (int32_t k = 0; k < n; ++k) w[k] = a[(size_t)ord[k] * n + ord[k]];
  int32_t *d_ord = d_sweeps + 1;  // kJacMax entries after the sweep count
  EIG_HIP(ctx, hipMemcpyAsync(d_ord, ord.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_gather_cols, dim3((unsigned)(((int64_t)n * n + 255) / 256)), dim3(256), 0,
                     st, V, (const double *)work, (const int32_t *)d_ord, n);
  EIG_HIP(ctx, hipGetLastError());
  EIG_HIP(ctx, hipStreamSynchronize(st));  // ord lives on this host frame
  return EIG_OK;
}

// Columns j < r of V scaled by 1 / sqrt(w_j) (device, column-major ld n).
__global__ void k_scale_cols(double *__restrict__ V, int32_t n, int32_t r,
                             const double *__restrict__ s) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * r) return;
  V[idx] *= s[idx / n];
}

// Axis j = blockIdx.x of Ev (row-major n x K) to unit norm with its largest-|.| component (the
// first on ties) positive, as row j of out.  The host's three passes over the
// strided values and their pageable copy took 1.4 ms more for 100,000 x 10, 0.9 for 20,011.
__global__ __launch_bounds__(1024) void k_fpca_vecs(const double *__restrict__ Ev, int32_t n, int32_t K,
                                                    double *__restrict__ out) {
  __shared__ double ss[1024], mx[1024];
  __shared__ int32_t at[1024];
  const int t = threadIdx.x;
  const double *x = Ev + blockIdx.x;
  double s = 0.0, m = -1.0;
  int32_t im = 0;
  for (int32_t i = t; i < n; i += 1024) {
    const double v = x[(int64_t)i * K];
    s += v * v;
    if (fabs(v) > m) {
      m = fabs(v);
      im = i;
    }
  }
  ss[t] = s;
  mx[t] = m;
  at[t] = im;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (t < o) {
      ss[t] += ss[t + o];
      if (mx[t + o] > mx[t] || (mx[t + o] == mx[t] && at[t + o] < at[t])) {
        mx[t] = mx[t + o];
        at[t] = at[t + o];
      }
    }
    __syncthreads();
  }
  const double f = (x[(int64_t)at[0] * K] < 0.0 ? -1.0 : 1.0) / sqrt(ss[0]);
  for (int32_t i = t; i < n; i += 1024) out[(int64_t)blockIdx.x * n + i] = f * x[(int64_t)i * K];
}

// X A in the split-BF16 form: A (npad x lda, rows = samples) split into the operands of
// cxa columns, then the persistent product into Y (rows = SNPs, ld ldy)
static int launch_xa_bf16(eig_ctx *ctx, const Plan &P, const uint32_t *lbf, uint16_t *frag,
                          int32_t cxa, const double *A, int32_t lda, double *Y, int64_t ldy, int32_t C,
                          hipStream_t st) {
  const int CT = cxa / 32;
  hipLaunchKernelGGL(k_fpca_split, dim3((unsigned)(P.npad / 32), (unsigned)CT), dim3(256), 0, st, A,
                     (int64_t)P.npad, (int64_t)lda, C, (int64_t)P.npad / 16, CT, frag);
  // four blocks a CU with 32 columns, two with 64 (their registers)
  const int64_t grid =
      std::min<int64_t>((P.M + 127) / 128, (int64_t)(CT == 1 ? 4 : 2) * std::max(ctx->num_cu, 1));
  hipLaunchKernelGGL((CT == 1 ? k_fpca_xa_bf16<1> : k_fpca_xa_bf16<2>), dim3((unsigned)grid), dim3(256),
                     0, st, P.sel, P.M, P.nst, lbf, (const uint16_t *)frag, Y, ldy, C, 4);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

// scale * X^T B in the split-BF16 form: B (M x ldb, rows = SNPs) split into the operands of
// its column groups; the SNP range is cut into S chunks (multiples of 64); the partials are
// summed in split order into out (ld ldo).  The result's rounding depends on the chunks, so
// they follow a fixed number of blocks per CU (three of 32 columns, two of 64), not the
// kernels' occupancy.
static int launch_xtb_bf16(eig_ctx *ctx, const Plan &P, const uint2 *selg, const uint32_t *tabs,
                           uint16_t *frag, int64_t Mpad, const double *B, int64_t ldb, int32_t C,
                           double *part, size_t part_doubles, double *out, int32_t ldo, double scale,
                           hipStream_t st) {
  // 32-column groups for a panel of up to 32 columns (the power iteration's at L <= 32),
  // else 64-column groups, which decode X^T once per 64 columns
  const int nct = C <= 32 ? 1 : 2, gw = 32 * nct;
  const int32_t ncg = (C + gw - 1) / gw, cp = gw * ncg;
  const int64_t slots = (int64_t)(nct == 1 ? 3 : 2) * std::max(ctx->num_cu, 1);
  hipLaunchKernelGGL(k_fpca_split, dim3((unsigned)(Mpad / 32), (unsigned)(cp / 32)), dim3(256), 0, st, B,
                     P.M, ldb, C, Mpad / 16, nct, frag);
  const int64_t G64 = Mpad / kGrp;
  const int64_t smax = std::max<int64_t>(
      1, std::min<int64_t>({64, G64, (int64_t)(part_doubles / ((size_t)P.npad * cp))}));
  int64_t chunk = Mpad, nsplit = 1;
  double best = -1.0;
  for (int64_t sp = 1; sp <= smax; ++sp) {
    int64_t c = (P.M + sp - 1) / sp;
    c = ((c + kGrp - 1) / kGrp) * kGrp;
    const int64_t ns = (P.M + c - 1) / c;
    if (ns != sp) continue;
    const double rounds = (double)((P.nst * ns * ncg + slots - 1) / slots);
    const double cost = rounds * (double)c / (double)P.M + 0.001 * (double)ns;
    if (best < 0.0 || cost < best - 1e-12) {
      best = cost;
      chunk = c;
      nsplit = ns;
    }
  }
  const int64_t items = (int64_t)P.nst * nsplit * ncg;
  hipLaunchKernelGGL((nct == 1 ? k_fpca_xtb_bf16<1> : k_fpca_xtb_bf16<2>), dim3((unsigned)items), dim3(256),
                     0, st, selg, G64, P.M, P.nst, tabs, (const uint16_t *)frag, (int32_t)nsplit, chunk, 8,
                     part, cp);
  const int64_t tot = (int64_t)P.npad * cp;
  hipLaunchKernelGGL(k_fpca_reduce, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st,
                     (const double *)part, (int32_t)nsplit, (int64_t)P.npad, cp, scale, out, ldo);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

extern "C" int eig_fpca(eig_ctx *ctx, int32_t K, int32_t L, int32_t I, uint64_t seed,
                        const double *omega, double *evals, double *evecs) {
  return eig_fpca_form(ctx, K, L, I, seed, omega, EIG_FORM_FP64, evals, evecs);
}

extern "C" int eig_fpca_form(eig_ctx *ctx, int32_t K, int32_t L, int32_t I, uint64_t seed,
                             const double *omega, int32_t form, double *evals, double *evecs) {
  if (!ctx || K <= 0 || L <= K || I <= 0 || !evals)
    return eig_set_err(ctx, EIG_E_ARG, "eig_fpca: need 0 < K < L and I > 0");
  if (form != EIG_FORM_FP64 && form != EIG_FORM_BF16X4)
    return eig_set_err(ctx, EIG_E_ARG, "eig_fpca: form must be FP64 or BF16X4");
  const bool bf = form == EIG_FORM_BF16X4;
  if (bf && L > 64) return eig_set_err(ctx, EIG_E_ARG, "eig_fpca: the BF16X4 form needs L <= 64");
  const int32_t Ctot = (I + 1) * L;
  if (L > 16 * kMaxCT || Ctot > kJacMax)
    return eig_set_err(ctx, EIG_E_ARG, "eig_fpca: L <= %d and (I+1)*L <= %d", 16 * kMaxCT,
                       kJacMax);
  if (!ctx->have_stats) return eig_set_err(ctx, EIG_E_STATE, "eig_fpca before eig_snpstats");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int64_t M = ctx->nsnp;
  const int32_t n = ctx->nrows, nst = ctx->nst, npad = nst * kTileS;
  // ncols: SNPs on the path (not removed by the caller's filters)
  std::vector<int32_t> status(M);
  EIG_HIP(ctx, hipMemcpy(status.data(), ctx->status.p, 4 * M, hipMemcpyDeviceToHost));
  int64_t ncols = 0;
  for (int64_t m = 0; m < M; ++m) ncols += status[m] != EIG_SNP_DEAD;
  if (ncols == 0) return eig_set_err(ctx, EIG_E_ARG, "eig_fpca: no SNPs");

  const int lda = 16 * ((L + 15) / 16);
  const int64_t ldq = ((Ctot + 15) / 16) * 16;
  const int Smax = 8;
  // workspace: lf | Omega x2 | Q | part | G | V | Vwork | U | B | small
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  size_t off = 0;
  auto add = [&](size_t b) {
    size_t o = off;
    off += up(b);
    return o;
  };
  const size_t o_lf = add(sizeof(double) * 4 * M);
  const size_t o_a0 = add(sizeof(double) * npad * lda), o_a1 = add(sizeof(double) * npad * lda);
  const size_t o_q = add(sizeof(double) * M * ldq);
  const size_t o_u = add(sizeof(double) * M * ldq);
  const size_t o_part = add(sizeof(double) * (size_t)Smax * npad * 16 * kMaxCT);
  const size_t o_b = add(sizeof(double) * npad * ldq);
  const size_t o_g = add(sizeof(double) * kJacMax * kJacMax);
  const size_t o_v = add(sizeof(double) * kJacMax * kJacMax);
  const size_t o_vw = add(sizeof(double) * kJacMax * kJacMax);
  const size_t o_sm = add(sizeof(double) * (kJacMax + 64) + sizeof(int32_t) * (kJacMax + 1));
  const size_t o_cb = add(sizeof(double) * kJacMax * kJacMax);
  const size_t o_ev = add(sizeof(double) * (size_t)K * npad);
  // split-BF16 form: levels, the X A panel (32 * ceil(L/32) columns) and the X^T B
  // panel (up to 64 * ceil(C/64) columns, C <= (I+1)L) as bf16 hi / lo operands, X^T B's
  // level tables
  const int64_t Mpad = ((M + kGrp - 1) / kGrp) * kGrp;
  const int32_t cxa = 32 * ((L + 31) / 32), cxb = 64 * ((Ctot + 63) / 64);
  const size_t o_lbf = bf ? add(sizeof(uint32_t) * 4 * M) : 0;
  const size_t o_ta = bf ? add(sizeof(uint16_t) * 2 * (size_t)cxa * npad) : 0;
  const size_t o_tb = bf ? add(sizeof(uint16_t) * 2 * (size_t)cxb * Mpad) : 0;
  const size_t o_tab = bf ? add(sizeof(uint32_t) * 2 * kFpTab * (size_t)(Mpad / kGrp)) : 0;
  // the split form reads all of the regrouped codes; without room for them the FP64 form's
  // products over SNPs take ranges of them
  bool released = false;
  EigInUse reads_selg(bf ? ctx->in_selg : released);
  const int rg = eig_ensure_selg(ctx);
  if (rg != EIG_OK && (bf || rg != EIG_E_NOMEM)) return rg;
  // FP64 form: the code products' digit operands and INT32 sums (codes.hip), one area for
  // the X A, X^T B and finishing X^T U products
  const int64_t G64 = Mpad / kGrp;
  FpcaPlans F{};
  size_t o_cw = 0;
  if (!bf) {
    F = eig_fpca_plans(ctx->num_cu, M, nst, K, L, Ctot);
    o_cw = add(F.area);
  }
  const CodesPlan &pa = F.pa, &pb = F.pb;
  EIG_TRY(eig_ensure(ctx, ctx->scratch2, off));
  char *base = (char *)ctx->scratch2.p;
  double *lf = (double *)(base + o_lf), *A0 = (double *)(base + o_a0), *A1 = (double *)(base + o_a1);
  double *Q = (double *)(base + o_q), *U = (double *)(base + o_u), *part = (double *)(base + o_part);
  double *Bm = (double *)(base + o_b), *G = (double *)(base + o_g), *V = (double *)(base + o_v);
  double *Vw = (double *)(base + o_vw), *sm = (double *)(base + o_sm), *Ev = (double *)(base + o_ev);
  int32_t *d_sweeps = (int32_t *)(sm + kJacMax);
  double *Cb = (double *)(base + o_cb);
  const size_t part_doubles = (size_t)Smax * npad * 16 * kMaxCT;
  uint32_t *lbf = bf ? (uint32_t *)(base + o_lbf) : nullptr;
  uint16_t *fa = bf ? (uint16_t *)(base + o_ta) : nullptr, *fb = bf ? (uint16_t *)(base + o_tb) : nullptr;
  uint32_t *tabs = bf ? (uint32_t *)(base + o_tab) : nullptr;

  eig_time_begin(ctx);
  hipLaunchKernelGGL(k_fpca_levels, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, st,
                     (const double *)ctx->mean.p, (const double *)ctx->fancy.p,
                     (const int32_t *)ctx->status.p, M, lf);
  if (omega) {
    std::vector<double> h((size_t)npad * lda, 0.0);
    for (int32_t i = 0; i < n; ++i)
      for (int32_t c = 0; c < L; ++c) h[(size_t)i * lda + c] = omega[(size_t)i * L + c];
    EIG_HIP(ctx, hipMemcpyAsync(A0, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice, st));
    EIG_HIP(ctx, hipStreamSynchronize(st));
  } else {
    const int64_t tot = (int64_t)npad * lda;
    hipLaunchKernelGGL(k_fpca_gauss, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, A0,
                       npad, lda, n, L, seed);
  }
  EIG_HIP(ctx, hipGetLastError());
  Plan P{M, nst, npad, (const uint32_t *)ctx->sel.p, lf};
  if (bf) {
    hipLaunchKernelGGL(k_fpca_levbf, dim3((unsigned)((4 * M + 255) / 256)), dim3(256), 0, st,
                       (const double *)lf, M, lbf);
    hipLaunchKernelGGL(k_fpca_tab, dim3((unsigned)(G64 * (kFpTab / 256))), dim3(256), 0, st,
                       (const uint32_t *)lbf, M, G64, tabs);
    EIG_HIP(ctx, hipGetLastError());
  }
  // X^T B and X A of the FP64 form, in the work area
  char *cw = base + o_cw;
  auto code_xtb = [&](const CodesPlan &plan, const double *B_, double scale, double *out, int64_t ldo,
                      int32_t Cpad) -> int {
    if (eig_codes_area(plan) > F.area) return eig_set_err(ctx, EIG_E_STATE, "eig_fpca: work area");
    CodeCols c{kColLevB, B_, ldq, M};
    c.lev = lf;
    return eig_codes_samples(ctx, plan, c, cw, npad, scale, out, ldo, 1, Cpad, st);
  };
  auto xa = [&](const double *A_, double *Y_) -> int {
    if (bf)
      return launch_xa_bf16(ctx, P, lbf, fa, cxa, A_, lda, Y_, ldq, L, st);
    const CodeCols c{kColPanel, A_, lda, n};
    char *sums = cw + pa.head_bytes + pa.dig_bytes;
    EIG_TRY(eig_codes_scales(ctx, pa, c, cw, st));
    EIG_TRY(eig_codes_build(ctx, pa, c, kCodeLinear, 0, cw, cw + pa.head_bytes, st));
    for (int64_t m = 0; m < M; m += F.arows) {
      const int64_t rows = std::min(F.arows, M - m);
      const CodeView v{(const uint8_t *)ctx->sel.p + m * 32, nullptr, 128 * 32, 32, M * 32, 16, rows,
                       (int64_t)nst * 8, kCodeLinear};
      EIG_HIP(ctx, eig_codes_product(pa, v, cw + pa.head_bytes, sums, false, st));
      EIG_TRY(eig_codes_out_pair(ctx, pa, rows, cw, sums, lf + 4 * m, nullptr, 1.0, Y_ + m * ldq, ldq, 1, st));
    }
    return EIG_OK;
  };
  auto xtb = [&](const double *B_, double *out_) -> int {
    if (bf)
      return launch_xtb_bf16(ctx, P, (const uint2 *)ctx->selg.p, tabs, fb, Mpad, B_, ldq, L,
                             part, part_doubles, out_, lda, 1.0 / (double)ncols, st);
    return code_xtb(pb, B_, 1.0 / (double)ncols, out_, lda, lda);
  };
  // ---- power iterations
  {
    double *cur = A0, *nxt = A1;
    for (int32_t i = 0; i < I; ++i) {
      EIG_TRY(xa(cur, Q + (size_t)i * L));
      EIG_TRY(xtb(Q + (size_t)i * L, nxt));
      std::swap(cur, nxt);
    }
    EIG_TRY(xa(cur, Q + (size_t)I * L));
  }
  EIG_HIP(ctx, hipGetLastError());
  eig_time_end(ctx, "fpca_power");

  // ---- orthonormal basis U of range(Q), block by block (kjg_fpca takes the SVD of
  // Q): each Krylov block is projected against the basis so far twice, orthonormalised
  // from its column-scaled Gram matrix, projected once more and orthonormalised again.
  // The blocks differ in scale by powers of the top eigenvalue, so one Gram matrix of
  // all of Q would lose the small directions that the SVD keeps.
  eig_time_begin(ctx);
  std::vector<double> w;
  int32_t r = 0;
  // W (nc columns, column-major nc x M at Wp, ld ldq) -= U_r (U_r^T W)
  auto project = [&](double *Wp, int32_t nc) -> int {
    if (r == 0) return EIG_OK;
    EIG_TRY(gemm_nt_long(ctx, !bf, r, nc, M, U, ldq, Wp, ldq, Cb, r, part, part_doubles, st));
    EIG_TRY(eig_gemm_f64(ctx, st, true, false, nc, M, r, -1.0, Cb, r, 0, U, ldq, 0, 1.0, Wp, ldq,
                         0, 1));
    return EIG_OK;
  };
  // Out (keep columns) = orthonormal basis of the nc columns at Wp
  auto orth = [&](const double *Wp, int32_t nc, double *Out, int32_t &keep) -> int {
    keep = 0;
    EIG_TRY(gemm_nt_long(ctx, !bf, nc, nc, M, Wp, ldq, Wp, ldq, G, nc, part, part_doubles, st));
    if (nc <= kJacLds) {
      hipLaunchKernelGGL(k_orth_lds, dim3(1), dim3(256), 0, st, (const double *)G, V, nc, 30, 1e-15,
                         d_sweeps);
      EIG_HIP(ctx, hipGetLastError());
      EIG_HIP(ctx, hipMemcpyAsync(&keep, d_sweeps, sizeof(int32_t), hipMemcpyDeviceToHost, st));
      EIG_HIP(ctx, hipStreamSynchronize(st));
      if (keep < 0) return eig_set_err(ctx, EIG_E_CONVERGE, "fpca: Jacobi did not converge");
      if (keep > 0)
        EIG_TRY(eig_gemm_f64(ctx, st, true, false, keep, M, nc, 1.0, V, nc, 0, Wp, ldq, 0, 0.0, Out,
                             ldq, 0, 1));
      return EIG_OK;
    }
    std::vector<double> g((size_t)nc * nc), dsc(nc);
    EIG_HIP(ctx, hipMemcpyAsync(g.data(), G, sizeof(double) * g.size(), hipMemcpyDeviceToHost, st));
    EIG_HIP(ctx, hipStreamSynchronize(st));
    for (int32_t i = 0; i < nc; ++i) {
      const double gi = g[(size_t)i * nc + i];
      dsc[i] = gi > 0.0 ? sqrt(gi) : 1.0;
    }
    for (int32_t jc = 0; jc < nc; ++jc)
      for (int32_t i = 0; i < nc; ++i) g[(size_t)jc * nc + i] /= dsc[i] * dsc[jc];
    EIG_HIP(ctx, hipMemcpyAsync(G, g.data(), sizeof(double) * g.size(), hipMemcpyHostToDevice, st));
    EIG_TRY(small_eigh(ctx, G, nc, V, w, Vw, d_sweeps));
    if (!(w[0] > 0.0)) return EIG_OK;
    while (keep < nc && w[keep] > 1e-13 * w[0]) ++keep;
    std::vector<double> v((size_t)nc * keep);
    EIG_HIP(ctx, hipMemcpyAsync(v.data(), V, sizeof(double) * v.size(), hipMemcpyDeviceToHost, st));
    EIG_HIP(ctx, hipStreamSynchronize(st));
    for (int32_t k = 0; k < keep; ++k)
      for (int32_t i = 0; i < nc; ++i) v[(size_t)k * nc + i] /= sqrt(w[k]) * dsc[i];
    EIG_HIP(ctx, hipMemcpyAsync(V, v.data(), sizeof(double) * v.size(), hipMemcpyHostToDevice, st));
    EIG_TRY(eig_gemm_f64(ctx, st, true, false, keep, M, nc, 1.0, V, nc, 0, Wp, ldq, 0, 0.0, Out,
                         ldq, 0, 1));
    return EIG_OK;
  };
  for (int32_t blk = 0; blk <= I; ++blk) {
    double *Ub = U + r, *Qb = Q + (size_t)blk * L;
    EIG_HIP(ctx, hipMemcpy2DAsync(Ub, sizeof(double) * ldq, Qb, sizeof(double) * ldq,
                                  sizeof(double) * L, (size_t)M, hipMemcpyDeviceToDevice, st));
    EIG_TRY(project(Ub, L));
    EIG_TRY(project(Ub, L));
    int32_t k1 = 0, k2 = 0;
    EIG_TRY(orth(Ub, L, Qb, k1));  // into the block's own (now free) columns of Q
    if (k1 == 0) continue;
    EIG_TRY(project(Qb, k1));
    EIG_TRY(orth(Qb, k1, Ub, k2));
    r += k2;
  }
  EIG_HIP(ctx, hipStreamSynchronize(st));
  const double *src = U;
  if (r < K) return eig_set_err(ctx, EIG_E_NUMERIC, "fpca: Krylov basis rank %d < K", r);
  // ---- B = X^T U  (npad x r, ld ldq), then the top-K left singular vectors of B
  if (bf) {
    // 64-column groups, and a remainder of at most 32 columns in a 32-column group, which
    // pads less (a 64-column group took 20 ms, a 32-column one 12 ms at N=100,000 x
    // M=500,000) when its 32 output columns stay within the row stride ldq
    const int32_t rem = r % 64;
    const int32_t r64 = (rem != 0 && rem <= 32 && r - rem + 32 <= ldq) ? r - rem : r;
    if (r64 > 0)
      EIG_TRY(launch_xtb_bf16(ctx, P, (const uint2 *)ctx->selg.p, tabs, fb, Mpad, src, ldq,
                              r64, part, part_doubles, Bm, (int32_t)ldq, 1.0, st));
    if (r64 < r)
      EIG_TRY(launch_xtb_bf16(ctx, P, (const uint2 *)ctx->selg.p, tabs, fb, Mpad, src + r64,
                              ldq, r - r64, part, part_doubles, Bm + r64, (int32_t)ldq, 1.0, st));
  } else {
    // planned for the rank that the basis has; the area holds the plan of every rank
    EIG_TRY(code_xtb(eig_fpca_basis_plan(ctx->num_cu, M, nst, r), src, 1.0, Bm, ldq, r));
  }
  EIG_TRY(gemm_nt_long(ctx, !bf, r, r, npad, Bm, ldq, Bm, ldq, G, r, part, part_doubles, st));
  // top-K eigenpairs of B^T B (order r up to 256) by the FP64 eigensolver: all
  // eigenvalues, K eigenvectors into V (column-major r x K)
  {
    std::vector<double> evh((size_t)K * r);
    w.assign(r, 0.0);
    EIG_TRY(eig_run_eigh(ctx, G, r, K, w.data(), evh.data(), true));
    EIG_HIP(ctx, hipMemcpyAsync(V, evh.data(), sizeof(double) * evh.size(), hipMemcpyHostToDevice,
                                st));
    EIG_HIP(ctx, hipStreamSynchronize(st));
  }
  std::vector<double> s(K);
  for (int32_t j = 0; j < K; ++j) {
    if (!(w[j] > 0.0)) return eig_set_err(ctx, EIG_E_NUMERIC, "fpca: singular value is zero");
    s[j] = 1.0 / sqrt(w[j]);
  }
  EIG_HIP(ctx, hipMemcpyAsync(sm, s.data(), sizeof(double) * K, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_scale_cols, dim3((unsigned)(((int64_t)r * K + 255) / 256)), dim3(256), 0,
                     st, V, r, K, (const double *)sm);
  // Ev (column-major K x npad == row-major npad x K) = V_K^T B^T
  EIG_TRY(eig_gemm_f64(ctx, st, true, false, K, npad, r, 1.0, V, r, 0, Bm, ldq, 0, 0.0, Ev, K, 0,
                       1));
  for (int32_t j = 0; j < K; ++j) evals[j] = w[j] / (double)ncols;  // S^2 / m (kjg_fpca.c:91-94)
  if (evecs) {
    // unit norm, largest-|.| component positive; Bm, which is free again, holds K rows of n
    hipLaunchKernelGGL(k_fpca_vecs, dim3((unsigned)K), dim3(1024), 0, st, (const double *)Ev, n, K, Bm);
    EIG_HIP(ctx, hipGetLastError());
  }
  eig_time_end(ctx, "fpca_finish");
  EigFetch f(ctx);
  EIG_TRY(f.get(evecs, Bm, sizeof(double) * (size_t)n * K));
  EIG_TRY(f.wait());
  return EIG_OK;
}
