// The FP64 form of XTX = Z^T Z on the integer matrix cores, exactly accumulated.
//
// A kept SNP's levels are f (g - mu) for genotype g (0 for a missing one), so with one
// side's factor f folded into the other
//     x_i x_j = [f x_i] (g_j - mu o_j),      o_j = 1 where sample j is observed, else 0.
// With q = rint(63 mu) and delta = mu - q/63 the right side splits into small integers:
//     x_i x_j = [f x_i / 63] (63 g_j - q o_j)  +  [-f x_i delta] o_j.
// Both brackets are written in fixed point with p1 and p2 balanced base-256 digits on
// one power-of-two grid, and every digit plane is multiplied with the integer plane of
// its term (63 g - q in [-126, 126], or o) by v_mfma_i32_32x32x32_i8.  The INT32 sums are
// exact (a chunk of SNPs is short enough for them), so the only rounding is that of the
// two brackets to their grids, relative to the panel's largest bracket, and of the final
// FP64 combination of the digits.
//
// A bracket's rounding error at a SNP is the same for every sample of that genotype, and o_j is
// 1 nearly everywhere, so row i of XTX would be off by the same sum of errors in every column,
// and column j, where most samples have the common genotype, in every row: harmless in an
// entry, but matrices of rank one, whose norm is the samples' number times that.  The errors
// are known where the digits are made.  With e1 and e2 the brackets' and b the integer that e1
// meets, their means over the samples marked by _,
//     sum e1_i b_j + e2_i o_j  =  sum (e1_i - e1_) b_ + (e2_i - e2_) o_  +  sum e1_ b_j + e2_ o_j  +  rest;
// k_xd_res forms the two sums, one for each sample as a row and one as a column, and k_xd_sum
// takes them out.  The rest differs in rows and columns.  Spectral norm of the error before and
// after, uncentred rare variants: 8.7e-12 and 1.1e-14 (198 samples x 2,000 SNPs), 2.8e-10 and
// 1.4e-14 (1,500 x 20,000).
//
// Measured against 80-bit sums over 2,000 to 300,000 SNPs, seven plus six digits leave 2 to 25 times less error than FP64 accumulation of
// the same products (an off-diagonal entry's rounding, 300,000 SNPs: 3.0e-12 against
// 8.0e-11; 2,000 SNPs: 1.3e-13 against 2.3e-13).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "eig_internal.h"

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4;
typedef __attribute__((__vector_size__(16 * sizeof(int)))) int i32x16;

namespace {
constexpr int kFrag = 1024;       // bytes of one MFMA operand: 32 samples x 32 SNPs
constexpr int kQ = 63;            // the grid of the right side's integers
constexpr int kXMaxP = 8;         // digits of the first bracket at most
constexpr int kXPlanes = 2 * kXMaxP + 2;

// ------------------------------------------------------------------ the panel's range
// max over SNPs and genotypes of |f level|, as the bits of a non-negative double (the
// order of such bits is the order of the values; a NaN compares above everything)
__global__ __launch_bounds__(256) void k_xd_max(const double *__restrict__ lev, int64_t M,
                                                unsigned long long *__restrict__ out) {
  double mx = 0.0;
  for (int64_t m = (int64_t)blockIdx.x * 256 + threadIdx.x; m < M; m += (int64_t)gridDim.x * 256) {
    const double *l = lev + 4 * m;
    const double l0 = l[0], l1 = l[1], l2 = l[2];
    const double f = fabs(0.5 * (l2 - l0));
    const double a = f * fmax(fmax(fabs(l0), fabs(l1)), fabs(l2));
    // fmax drops a NaN: keep it as an infinity
    mx = fmax(mx, isfinite(l0) && isfinite(l1) && isfinite(l2) ? a : INFINITY);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0)
    atomicMax(out, (unsigned long long)__double_as_longlong(mx));
}

// ------------------------------------------------------------------ digit tables
// tab[plane][k] for the chunk's SNP k: the plane's byte for codes 0, 1, 2 and 3 (missing:
// always 0), lowest byte first.  Planes: p1 digits of f x / 63 (highest first), p2 digits
// of -f x delta, 63 g - q, o.  SNPs past M and dropped ones are all zero.  res[k][code]: the
// share of a sample of that code in the left-out parts of its row (x) and its column (y); the
// means take genotype frequencies from the allele's, which is near enough.
__global__ __launch_bounds__(256) void k_xd_tab(const double *__restrict__ lev, int64_t m0,
                                                int64_t M, int64_t K, int32_t p1, int32_t p2,
                                                double s1, double s2, const int32_t *__restrict__ c0,
                                                const int32_t *__restrict__ c1, const int32_t *__restrict__ nmiss,
                                                int32_t nrows, uint32_t *__restrict__ tab,
                                                double2 *__restrict__ res) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= K) return;
  const int64_t m = m0 + k;
  double l[3] = {0.0, 0.0, 0.0};
  if (m < M)
#pragma unroll
    for (int g = 0; g < 3; ++g) l[g] = lev[4 * m + g];
  const double f = 0.5 * (l[2] - l[0]);
  const double mu = f != 0.0 ? -l[0] / f : 0.0;
  const double q = rint((double)kQ * mu);
  const double delta = mu - q / (double)kQ;
  int64_t a1[3], a2[3];
  double seen = 0.0, p = 0.0;
  if (m < M) {
    seen = 1.0 - (double)nmiss[m] / (double)nrows;
    p = (double)c0[m] / fmax(1.0, (double)c0[m] + (double)c1[m]);
  }
  double e1[3], e2[3];
#pragma unroll
  for (int g = 0; g < 3; ++g) {
    const double a = f * l[g], b = -a * delta;
    a1[g] = llrint(a / (double)kQ * s1);
    a2[g] = llrint(b * s2);
    // both left-out parts without a rounding of their own that matters: a fused product's
    e1[g] = fma(-(double)kQ, (double)a1[g] / s1, a) / (double)kQ;
    e2[g] = (b - (double)a2[g] / s2) + fma(-a, delta, -b);
  }
  auto mean = [&](const double (&e)[3]) {
    return seen * ((1.0 - p) * ((1.0 - p) * e[0] + 2.0 * p * e[1]) + p * p * e[2]);
  };
  const double m1 = mean(e1), m2 = mean(e2), bm = seen * ((double)kQ * delta);
#pragma unroll
  for (int g = 0; g < 3; ++g)
    res[4 * k + g] = make_double2((e1[g] - m1) * bm + (e2[g] - m2) * seen, m1 * ((double)(kQ * g) - q) + m2);
  res[4 * k + 3] = make_double2(-m1 * bm - m2 * seen, 0.0);
  auto digits = [&](int64_t (&v)[3], int32_t p, int32_t base) {
    for (int32_t s = p - 1; s >= 0; --s) {  // lowest digit first
      uint32_t w = 0;
#pragma unroll
      for (int g = 0; g < 3; ++g) {
        const int32_t d = (int8_t)(v[g] & 0xFF);
        v[g] = (v[g] - d) >> 8;
        w |= ((uint32_t)d & 0xFFu) << (8 * g);
      }
      tab[(int64_t)(base + s) * K + k] = w;
    }
  };
  digits(a1, p1, 0);
  digits(a2, p2, p1);
  uint32_t wb = 0, wo = 0;
  if (f != 0.0)
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      wb |= ((uint32_t)(kQ * g - (int32_t)q) & 0xFFu) << (8 * g);
      wo |= 1u << (8 * g);
    }
  tab[(int64_t)(p1 + p2) * K + k] = wb;
  tab[(int64_t)(p1 + p2 + 1) * K + k] = wo;
}

// part[split][sample]: the sums of res over a split's SNPs (of the chunk's, kResSnps at a time) for
// the 128 samples of a tile: thread (s, w) of a block adds the 16 samples of word w at every
// 32nd SNP.  A pass over the codes with an LDS lookup of 16 bytes each, which is what bounds
// it: 0.14 ms for 5,000 samples x 100,000 SNPs (58 TB/s of LDS), where the product takes 14.7.
__global__ __launch_bounds__(256) void k_xd_res(const uint32_t *__restrict__ sel, int64_t M, int64_t m0,
                                                int64_t K, int32_t nstep, const double2 *__restrict__ res,
                                                double2 *__restrict__ part) {
  __shared__ __align__(16) double2 tab[kResSnps][4];
  __shared__ __align__(16) double2 red[32][kTileS / 4 + 1], half[8][kTileS / 4];
  const int t = threadIdx.x, w = t & 7, s = t >> 3;
  const int32_t tile = blockIdx.x;
  double2 acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = make_double2(0.0, 0.0);
  for (int32_t b = 0; b < nstep; ++b) {
    const int64_t k0 = ((int64_t)blockIdx.y * nstep + b) * kResSnps;
    if (k0 >= K) break;  // uniform
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kResSnps / 64; ++u) {
      const int64_t k = k0 + (t >> 2) + 64 * u;
      tab[(t >> 2) + 64 * u][t & 3] = k < K ? res[4 * k + (t & 3)] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    uint32_t x[kResSnps / 32];
#pragma unroll
    for (int u = 0; u < kResSnps / 32; ++u) {
      const int64_t m = m0 + k0 + s + 32 * u;
      x[u] = m < M ? sel[((int64_t)tile * M + m) * kTileWords + w] : ~0u;
    }
#pragma unroll
    for (int u = 0; u < kResSnps / 32; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const double2 e = tab[s + 32 * u][(x[u] >> (2 * i)) & 3u];
        acc[i].x += e.x;
        acc[i].y += e.y;
      }
  }
  // four of each word's samples at a time
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) red[s][4 * w + i] = acc[4 * q + i];
    __syncthreads();
    const int j = t & 31, h = t >> 5;
    double2 v = make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v.x += red[4 * h + u][j].x;
      v.y += red[4 * h + u][j].y;
    }
    half[h][j] = v;
    __syncthreads();
    if (t < kTileS / 4) {
#pragma unroll
      for (int u = 1; u < 8; ++u) {
        v.x += half[u][t].x;
        v.y += half[u][t].y;
      }
      part[((int64_t)blockIdx.y * gridDim.x + tile) * kTileS + 16 * (t >> 2) + 4 * q + (t & 3)] = v;
    }
  }
}
// out[i] = sum of the splits' parts
__global__ __launch_bounds__(256) void k_xd_res_sum(const double2 *__restrict__ part, int32_t nsplit,
                                                    int32_t n, double2 *__restrict__ out) {
  __shared__ __align__(16) double2 red[16][16];
  const int j = threadIdx.x & 15, h = threadIdx.x >> 4;
  const int32_t i = blockIdx.x * 16 + j;  // n is a multiple of 128
  double2 v = make_double2(0.0, 0.0);
#pragma unroll 4
  for (int32_t s = h; s < nsplit; s += 16) {
    const double2 e = part[(int64_t)s * n + i];
    v.x += e.x;
    v.y += e.y;
  }
  red[h][j] = v;
  __syncthreads();
  if (h != 0) return;
  for (int u = 1; u < 16; ++u) {
    v.x += red[u][j].x;
    v.y += red[u][j].y;
  }
  out[i] = v;
}

// ------------------------------------------------------------------ operand planes
// planes[((plane * RT + rt) * KS + ks) * 1024 ..]: the MFMA operand of samples 32 rt ..
// and SNPs 32 ks .. of the chunk, lane l's 16 bytes at 16 l: sample l % 32, SNPs
// 16 (l / 32) + 0 .. 15.  One wave builds the operands of all planes for two row tiles:
// the 4 x 16 codes of a lane become byte selectors once, and each plane is then three
// byte permutes per four SNPs of its table words, which all lanes of a half share.
__global__ __launch_bounds__(256) void k_xd_planes(const uint32_t *__restrict__ sel, int64_t M,
                                                   int32_t nst, int64_t m0, int64_t K,
                                                   int32_t np, int32_t RT,
                                                   const uint32_t *__restrict__ tab,
                                                   uint8_t *__restrict__ planes) {
  __shared__ __align__(16) uint32_t st[kXPlanes][32];
  __shared__ uint32_t words[32][kTileWords];
  const int64_t KS = K / 32;
  const int64_t ks = blockIdx.x;
  const int32_t tile = blockIdx.y;  // 128 samples: row tiles 4 tile .. 4 tile + 3
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  for (int e = t; e < np * 32; e += 256) st[e >> 5][e & 31] = tab[(int64_t)(e >> 5) * K + ks * 32 + (e & 31)];
  {
    const int64_t m = m0 + ks * 32 + (t >> 3);
    words[t >> 3][t & 7] = (tile < nst && m < M) ? sel[((int64_t)tile * M + m) * kTileWords + (t & 7)] : ~0u;
  }
  __syncthreads();
  const int row = 32 * w + (lane & 31), h = lane >> 5;
  uint32_t s01[4], s23[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    uint32_t c[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) c[b] = (words[16 * h + 4 * u + b][row >> 4] >> (2 * (row & 15))) & 3u;
    // v_perm_b32(hi, lo, s): selector bytes 0-3 pick from lo, 4-7 from hi
    s01[u] = c[0] | ((c[1] + 4u) << 8);
    s23[u] = c[2] | ((c[3] + 4u) << 8);
  }
  uint8_t *dst = planes + (((int64_t)4 * tile + w) * KS + ks) * kFrag + lane * 16;
  const int64_t pstep = (int64_t)RT * KS * kFrag;
  for (int p = 0; p < np; ++p) {
    uint32_t o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint4 tw = *(const uint4 *)&st[p][16 * h + 4 * u];
      const uint32_t a = __builtin_amdgcn_perm(tw.y, tw.x, s01[u]);
      const uint32_t b = __builtin_amdgcn_perm(tw.w, tw.z, s23[u]);
      o[u] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    }
    *(uint4 *)(dst + p * pstep) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// ------------------------------------------------------------------ the product
// One block per (split, digit, tile pair): 256 x 256 INT32 sums over the split's SNPs of
// digit plane s of the first bracket with 63 g - q, then of the second's with o.  64 SNPs
// (32 KB) per LDS stage, three stages, the loads of a stage issued two stages before its
// stores; a wave reads the next operands from LDS while the current MFMAs run.
// Four waves of 128 x 128, one per SIMD with 384 registers: LDS traffic bounds smaller
// wave tiles (eight waves of 128 x 64 read 96 and write 32 bytes per CU cycle of MFMA at
// full rate, the LDS' own 128; here it is 94).  At 5,000 samples x 600,000 SNPs,
// six chunks of 13 products: 14.7 ms a chunk, 2.4 POP/s, the matrix units busy 72 % of the
// cycles at the clock that this load leaves, 1.6 GHz (chunks of 120,000 SNPs took 17.7 ms,
// and an eight-wave kernel 19.5 scheduled alike, 21 without the interleaving below).
struct XdArgs {
  const uint8_t *planes;
  const uint32_t *pairs;  // tile pair list: row tile | column tile << 16
  int32_t *part;          // [split][digit][pair][256 * 256]
  int64_t KS;             // 32-SNP steps in the chunk (a multiple of 4)
  int32_t RT, npair, p1, p2, nsplit;
  int32_t per;            // 64-SNP stages per split (even)
};

__global__ __launch_bounds__(256, 1) void k_xd_gemm(XdArgs A) {
  __shared__ __align__(16) uint8_t lds[3][2][8 * 2 * kFrag];
  // consecutive items run on one XCD (blocks go to the eight XCDs in turn), so that the
  // tile pairs of a band share their strips in its L2
  const int64_t items = (int64_t)A.npair * A.p1 * A.nsplit;
  const int64_t per8 = (items + 7) / 8;
  const int64_t item = (int64_t)(blockIdx.x & 7) * per8 + (blockIdx.x >> 3);
  if ((int64_t)(blockIdx.x >> 3) >= per8 || item >= items) return;
  const int32_t pr = (int32_t)(item % A.npair);
  const int32_t s = (int32_t)((item / A.npair) % A.p1);
  const int32_t split = (int32_t)(item / ((int64_t)A.npair * A.p1));
  const uint32_t pw = A.pairs[pr];
  const int32_t ti = pw & 0xFFFF, tj = pw >> 16;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, wr = w >> 1, wc = w & 1;
  const int32_t nstage = (int32_t)(A.KS / 2);
  const int32_t k0 = split * A.per, n0 = min(A.per, nstage - k0);
  const int32_t ntot = s < A.p2 ? 2 * n0 : n0;
  const int64_t strip = A.KS * kFrag, pl = (int64_t)A.RT * strip;
  const uint8_t *a1 = A.planes + s * pl + (int64_t)ti * 8 * strip + (int64_t)k0 * 2 * kFrag;
  const uint8_t *a2 = A.planes + (A.p1 + (s < A.p2 ? s : 0)) * pl + (int64_t)ti * 8 * strip +
                      (int64_t)k0 * 2 * kFrag;
  const uint8_t *b1 = A.planes + (int64_t)(A.p1 + A.p2) * pl + (int64_t)tj * 8 * strip +
                      (int64_t)k0 * 2 * kFrag;
  const uint8_t *b2 = b1 + pl;
  int64_t vo[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) vo[u] = (int64_t)((t >> 7) + 2 * u) * strip + (t & 127) * 16;
  auto load = [&](int32_t g, i32x4 (&r)[8]) {
    const int32_t gc = min(g, ntot - 1);
    const bool second = gc >= n0;
    const uint8_t *pa = second ? a2 + (int64_t)(gc - n0) * (2 * kFrag) : a1 + (int64_t)gc * (2 * kFrag);
    const uint8_t *pb = second ? b2 + (int64_t)(gc - n0) * (2 * kFrag) : b1 + (int64_t)gc * (2 * kFrag);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      r[u] = *(const i32x4 *)(pa + vo[u]);
      r[4 + u] = *(const i32x4 *)(pb + vo[u]);
    }
  };
  auto store = [&](int buf, const i32x4 (&r)[8]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      *(i32x4 *)&lds[buf][0][4096 * u + t * 16] = r[u];
      *(i32x4 *)&lds[buf][1][4096 * u + t * 16] = r[4 + u];
    }
  };
  auto frag = [&](int buf, int ks, i32x4 (&fa)[4], i32x4 (&fb)[4]) {
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      fb[y] = *(const i32x4 *)&lds[buf][1][((4 * wc + y) * 2 + ks) * kFrag + lane * 16];
      fa[y] = *(const i32x4 *)&lds[buf][0][((4 * wr + y) * 2 + ks) * kFrag + lane * 16];
    }
  };
  i32x16 acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0;
  auto mma = [&](const i32x4 (&fa)[4], const i32x4 (&fb)[4]) {
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y)
        acc[x][y] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[x], fb[y], acc[x][y], 0, 0, 0);
  };
  i32x4 r0[8], r1[8];
  load(0, r0);
  load(1, r1);
  store(0, r0);
  load(2, r0);
  store(1, r1);
  __syncthreads();
  i32x4 fa0[4], fb0[4], fa1[4], fb1[4];
  frag(0, 0, fa0, fb0);
  int b = 0;
  auto step = [&](int32_t g, i32x4 (&rn)[8], i32x4 (&rs)[8]) {
    const int bn = b == 2 ? 0 : b + 1, bs = bn == 2 ? 0 : bn + 1;
    frag(b, 1, fa1, fb1);
    load(g + 3, rn);
    mma(fa0, fb0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    store(bs, rs);
    frag(bn, 0, fa0, fb0);
    mma(fa1, fb1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    b = bn;
  };
  for (int32_t g = 0; g < ntot; g += 2) {
    step(g, r1, r0);
    step(g + 1, r0, r1);
  }
  int32_t *out = A.part + (((int64_t)split * A.p1 + s) * A.npair + pr) * (kXT * kXT);
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 128 * wr + 32 * x + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int col = 128 * wc + 32 * y + (lane & 31);
        out[row * kXT + col] = acc[x][y][r];
      }
}

// ------------------------------------------------------------------ the digits' sum
// dst (128 x 128 FP64 lower tiles, tile pair (i, j) at i (i + 1) / 2 + j): the chunk's sum
// over splits (exact) and digits (Horner, FP64), times the grid, and the left-out parts of
// its row and column, added to the earlier chunks' unless this is the first.  16 blocks per
// quarter of a 256 x 256 pair.
__global__ __launch_bounds__(256) void k_xd_sum(const int32_t *__restrict__ part,
                                                const uint32_t *__restrict__ pairs, int32_t npair,
                                                int32_t p1, int32_t nsplit, int32_t nst,
                                                double grid, int32_t first,
                                                const double2 *__restrict__ res, int32_t nres,
                                                double *__restrict__ dst) {
  const int32_t pr = blockIdx.x >> 6, qd = (blockIdx.x >> 4) & 3, slab = blockIdx.x & 15;
  const uint32_t pw = pairs[pr];
  const int32_t i = 2 * (pw & 0xFFFF) + (qd >> 1), j = 2 * (pw >> 16) + (qd & 1);
  if (i >= nst || j > i) return;
  // 8 rows of 128: thread t holds 4 columns of row t / 32
  const int r = slab * 8 + (threadIdx.x >> 5), c = (threadIdx.x & 31) * 4;
  const int64_t e = (int64_t)((qd >> 1) * 128 + r) * kXT + (qd & 1) * 128 + c;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  for (int32_t s = 0; s < p1; ++s) {
    int64_t a[4] = {0, 0, 0, 0};
#pragma unroll 8
    for (int32_t sp = 0; sp < nsplit; ++sp) {
      const i32x4 x = *(const i32x4 *)(part + (((int64_t)sp * p1 + s) * npair + pr) * (kXT * kXT) + e);
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] += x[u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = v[u] * 256.0 + (double)a[u];
  }
  double *o = dst + ((int64_t)i * (i + 1) / 2 + j) * (kTileS * kTileS) + r * kTileS + c;
  double row = 0.0, col[4] = {0.0, 0.0, 0.0, 0.0};
  for (int32_t s = 0; s < nres; ++s) {
    const double2 *e = res + (int64_t)s * nst * kTileS;
    row += e[i * kTileS + r].x;
#pragma unroll
    for (int u = 0; u < 4; ++u) col[u] += e[j * kTileS + c + u].y;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const double x = v[u] * grid + (row + col[u]);
    o[u] = first ? x : o[u] + x;
  }
}
}  // namespace

// The lower 128 x 128 tiles of XTX into dst (tile pair (i, j) at i (i + 1) / 2 + j).
// *done = 0 when the workspace does not fit the card or the panel's levels are outside
// the scheme's range (neither finite nor within 2^+-200: no normalisation gives such).
int eig_syrk_digits(eig_ctx *ctx, double *dst, int *done) {
  *done = 0;
  const int64_t M = ctx->nsnp;
  const int32_t nst = ctx->nst;
  hipStream_t st = ctx->stream;
  const double *lev = (const double *)ctx->lev.p;
  const int32_t nT = (nst + 1) / 2, npair = nT * (nT + 1) / 2;
  // tile pairs in bands of four rows, column by column: 32 consecutive pairs touch
  // about four row strips and eight column strips
  std::vector<uint32_t> pairs;
  for (int32_t b = 0; b < nT; b += 4)
    for (int32_t j = 0; j < std::min(b + 4, nT); ++j)
      for (int32_t i = std::max(b, j); i < std::min(b + 4, nT); ++i)
        pairs.push_back((uint32_t)i | ((uint32_t)j << 16));
  EIG_TRY(eig_ensure(ctx, ctx->xdmisc, 256 + 4 * (size_t)npair));
  unsigned long long *d_max = (unsigned long long *)ctx->xdmisc.p;
  uint32_t *d_pairs = (uint32_t *)ctx->xdmisc.p + 64;
  EIG_HIP(ctx, hipMemsetAsync(d_max, 0, 8, st));
  hipLaunchKernelGGL(k_xd_max, dim3((unsigned)std::min<int64_t>((M + 255) / 256, 1024)), dim3(256), 0,
                     st, lev, M, d_max);
  EIG_HIP(ctx, hipGetLastError());
  unsigned long long bits = 0;
  EIG_HIP(ctx, hipMemcpyAsync(&bits, d_max, 8, hipMemcpyDeviceToHost, st));
  EIG_HIP(ctx, hipMemcpyAsync(d_pairs, pairs.data(), 4 * (size_t)npair, hipMemcpyHostToDevice, st));
  EIG_HIP(ctx, hipStreamSynchronize(st));
  double mx;
  std::memcpy(&mx, &bits, 8);
  if (!std::isfinite(mx)) return EIG_OK;
  int E = -200;
  if (mx > 0.0) E = (int)std::ceil(std::log2(mx / kQ * 1.01));
  if (mx > 0.0 && (E < -200 || E > 200)) return EIG_OK;
  // digits: the brackets' rounding, ~1.4e-15 2^E sqrt(M) per entry with seven plus six of
  // them and ~2.9e-16 2^E sqrt(M) with seven plus seven, stays below the FP64 product's
  // own, which is at least ~1.2e-16 M (all three measured against 80-bit sums on panels
  // of 2,000 to 300,000 SNPs with E from 1 to 7); eight plus seven leave less than either
  const double r = std::ldexp(1.0, E) / std::sqrt((double)M);
  const int32_t p1 = r <= 0.4 ? 7 : 8, p2 = r <= 0.08 ? 6 : 7;
  const XdPlan X = eig_xd_plan(ctx->num_cu, M, nst, p1, p2);
  const int32_t np = X.np, RT = X.RT;
  const int64_t K = X.K;
  if (eig_ensure(ctx, ctx->xdplanes, X.plane_bytes) != EIG_OK ||
      eig_ensure(ctx, ctx->xdtab, X.tab_bytes) != EIG_OK ||
      eig_ensure(ctx, ctx->xdpart, X.part_bytes) != EIG_OK) {
    for (DevBuf *b : {&ctx->xdplanes, &ctx->xdtab, &ctx->xdpart}) {
      if (b->p) hipFree(b->p);
      *b = DevBuf();
    }
    return EIG_OK;
  }
  // [K][4], the splits' sums, the chunk's sums, the digit tables
  double2 *d_res = (double2 *)ctx->xdtab.p;
  double2 *d_rpart = d_res + 4 * K, *d_rsum = d_rpart + (size_t)X.rsplit * nst * kTileS;
  uint32_t *d_tab = (uint32_t *)(d_rsum + (size_t)nst * kTileS);
  const double s1 = std::ldexp(1.0, 8 * p1 - 1 - E), s2 = std::ldexp(1.0, 8 * p2 - 1 - E);
  const double grid = std::ldexp(1.0, E + 1 - 8 * p1);
  for (int64_t c = 0; c < X.nchunk; ++c) {
    const int64_t m0 = c * K;
    hipLaunchKernelGGL(k_xd_tab, dim3((unsigned)((K + 255) / 256)), dim3(256), 0, st, lev, m0, M, K, p1,
                       p2, s1, s2, (const int32_t *)ctx->c0.p, (const int32_t *)ctx->c1.p,
                       (const int32_t *)ctx->nmiss.p, ctx->nrows, d_tab, d_res);
    hipLaunchKernelGGL(k_xd_res, dim3((unsigned)nst, (unsigned)X.rsplit), dim3(256), 0, st,
                       (const uint32_t *)ctx->sel.p, M, m0, K, X.rstep, (const double2 *)d_res, d_rpart);
    // few splits are added up by k_xd_sum itself, which saves a launch, while its blocks are
    // one round of the device: each adds them up again
    const bool few = X.rsplit <= 16 && npair * 64 <= ctx->num_cu;
    if (!few)
      hipLaunchKernelGGL(k_xd_res_sum, dim3((unsigned)(nst * kTileS / 16)), dim3(256), 0, st,
                         (const double2 *)d_rpart, X.rsplit, nst * kTileS, d_rsum);
    hipLaunchKernelGGL(k_xd_planes, dim3((unsigned)(K / 32), (unsigned)(RT / 4)), dim3(256), 0, st,
                       (const uint32_t *)ctx->sel.p, M, nst, m0, K, np, RT,
                       (const uint32_t *)d_tab, (uint8_t *)ctx->xdplanes.p);
    for (int32_t b = 0; b < npair; b += X.band) {
      const int32_t nb = std::min(X.band, npair - b);
      const XdArgs A{(const uint8_t *)ctx->xdplanes.p, d_pairs + b, (int32_t *)ctx->xdpart.p, K / 32, RT, nb,
                     p1, p2, X.nsplit, X.per};
      const int64_t items = (int64_t)nb * p1 * X.nsplit;
      hipLaunchKernelGGL(k_xd_gemm, dim3((unsigned)((items + 7) / 8 * 8)), dim3(256), 0, st, A);
      hipLaunchKernelGGL(k_xd_sum, dim3((unsigned)nb * 64), dim3(256), 0, st, (const int32_t *)ctx->xdpart.p,
                         d_pairs + b, nb, p1, X.nsplit, nst, grid, (int32_t)(c == 0),
                         (const double2 *)(few ? d_rpart : d_rsum), few ? X.rsplit : 1, dst);
    }
    EIG_HIP(ctx, hipGetLastError());
  }
  *done = 1;
  return EIG_OK;
}
