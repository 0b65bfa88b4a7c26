// Products of packed genotype codes with FP64 columns on the integer matrix cores.
//
// With a sample's genotype at a SNP written as its 2-bit code c (3 = missing) and the
// missing bit m, every normalised value is linear in the two:
//     x = f (c - 3 m) + l0 (1 - m),
// f and l0 the SNP's scale and its level of genotype 0.  A sum over k of x_rk B_kj is then
//     sum c (f B) - sum m (3 f + l0) B + sum l0 B     (k = SNPs, factors into the columns)
//     f (sum c A - 3 sum m A) + l0 (sum A - sum m A)  (k = samples, factors on the result),
// products of small integers with FP64 columns.  Each column is written in fixed point
// with seven balanced base-256 digits under the power of two above its largest entry (its
// entries within 2^-54 of that), and c and m (bytes 0-3 and 0-1, three shifts and masks
// from a code word) are multiplied with the digit planes by v_mfma_i32_16x16x64_i8.  The
// INT32 sums are exact, so the result has no rounding but the grid's and the final
// conversion's: less than FP64 accumulation leaves, and the same bits however the sums are
// split.
//
// Used by fastmode's FP64 panel products (kjg_fpca.c:104-178), the SNP loadings and their
// scales (smartpca.c:1438-1525) and lsqproject's normal equations (smartpca.c:4606-4757).
#include <algorithm>
#include <cmath>

#include "eig_internal.h"

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4;
typedef unsigned long long u64;

namespace {
constexpr int kDig = 7;      // digits per column
constexpr int kSt = 128;     // k per stage
constexpr int kFragB = 1024;  // bytes of a digit operand: 16 digit columns x 64 k
constexpr int kMaxCols = 20;  // columns of a group of nine tiles (140 of 144 digit columns)
constexpr int kMaxNT = 9;

// ------------------------------------------------------------------ columns
// The three FP64 values of column c at index k: v1 multiplies the code, v2 the missing
// bit, v3 is summed alone.
struct ColArgs {
  const double *a;      // panel, axes or loadings
  int64_t ld;           // their leading dimension
  int64_t n;            // valid k: 0 .. n-1
  const double *lev;    // lev[k][4], or
  const double *fancy, *xmean;  // scale and -l0, with
  const uint8_t *ignore;        // SNPs that read as absent
  const double *fxscal;
  int32_t K;            // lsqproject's axes
};
struct Col3 {
  double v1, v2, v3;
};
// column p of the Gram's upper triangle, by rows
__device__ __forceinline__ void tri_pair(int32_t p, int32_t K, int32_t &a, int32_t &b) {
  a = 0;
  while (p >= K - a) {
    p -= K - a;
    ++a;
  }
  b = a + p;
}
template <int KIND>
__device__ __forceinline__ Col3 col_value(const ColArgs &A, int64_t k, int32_t c) {
  Col3 v{0.0, 0.0, 0.0};
  if (k >= A.n) return v;
  if constexpr (KIND == kColPanel) {  // row-major panel, samples
    v.v1 = v.v2 = v.v3 = A.a[k * A.ld + c];
  } else if constexpr (KIND == kColAxes) {  // column-major, samples
    v.v1 = v.v2 = v.v3 = A.a[(int64_t)c * A.ld + k];
  } else if constexpr (KIND == kColLevB) {  // row-major panel over SNPs, level table
    const double l0 = A.lev[4 * k], f = 0.5 * (A.lev[4 * k + 2] - l0), b = A.a[k * A.ld + c];
    v.v1 = f * b;
    v.v2 = -(3.0 * f + l0) * b;
    v.v3 = l0 * b;
  } else if constexpr (KIND == kColFx) {  // loadings, column-major over SNPs
    if (!A.ignore[k]) {
      const double f = A.fancy[k], xm = A.xmean[k], b = A.a[(int64_t)c * A.ld + k];
      v.v1 = f * b;
      v.v2 = (xm - 3.0 * f) * b;
      v.v3 = -xm * b;
    }
  } else if constexpr (KIND == kColLsqR) {  // right-hand sides, then the observed count
    if (!A.ignore[k] && c == A.K) {
      v.v2 = -1.0;
      v.v3 = 1.0;
    } else if (!A.ignore[k]) {
      const double f = A.fancy[k], xm = A.xmean[k], b = A.fxscal[c] * A.a[(int64_t)c * A.ld + k];
      v.v1 = f * b;
      v.v2 = (xm - 3.0 * f) * b;
      v.v3 = -xm * b;
    }
  } else {  // kColLsqG: the Gram's products, on observed SNPs
    if (!A.ignore[k]) {
      int32_t i, j;
      tri_pair(c, A.K, i, j);
      const double p =
          (A.fxscal[i] * A.a[(int64_t)i * A.ld + k]) * (A.fxscal[j] * A.a[(int64_t)j * A.ld + k]);
      v.v2 = -p;
      v.v3 = p;
    }
  }
  return v;
}

// the element that code slot i of word j (of a stage's eight, from word j0) holds
__device__ __forceinline__ int64_t code_elem(int32_t layout, int64_t j, int32_t i) {
  if (layout == kCodeLinear) return 16 * j + i;
  if (layout == kCodeGrouped) {  // selg: see eig_ensure_selg
    const int64_t g = j >> 2;
    const int32_t w = (int32_t)(j & 3);
    return 64 * g + 16 * (2 * (w & 1) + (i >> 3)) + 8 * (w >> 1) + (i & 7);
  }
  return 16 * j + 4 * (i >> 2) + 3 - (i & 3);  // kCodeBytes: the first of a byte in its top bits
}

__global__ void k_cd_zero(u64 *__restrict__ p, int32_t n) {
  const int32_t i = (int32_t)(blockIdx.x * 256 + threadIdx.x);
  if (i < n) p[i] = 0;
}

// mx[c]: max over k of |v1|, |v2|, |v3| as the bits of a double (NaN above all).  Threads
// keep one column each; row-major panels are read a row at a time, others along k.
template <int KIND>
__global__ __launch_bounds__(256) void k_cd_max(ColArgs A, int64_t k1, int32_t C, u64 *__restrict__ mx) {
  constexpr bool rowmajor = KIND == kColPanel || KIND == kColLevB;
  __shared__ u64 red[256];
  u64 m = 0;
  int32_t c;
  const int t = threadIdx.x;
  auto up = [&](int64_t k) {
    const Col3 v = col_value<KIND>(A, k, c);
    const double a[3] = {fabs(v.v1), fabs(v.v2), fabs(v.v3)};
#pragma unroll
    for (int u = 0; u < 3; ++u) m = max(m, (u64)__double_as_longlong(a[u]));
  };
  red[t] = 0;
  __syncthreads();
  if constexpr (rowmajor) {
    const int32_t w = min(C, 256), rows = 256 / w;
    for (int32_t c0 = 0; c0 < C; c0 += w) {
      c = c0 + t % w;
      m = 0;
      if (t < rows * w && c < C)
        for (int64_t k = (int64_t)blockIdx.x * rows + t / w; k < k1; k += (int64_t)gridDim.x * rows) up(k);
      if (t < rows * w && c < C) atomicMax(&red[t % w], m);
      __syncthreads();
      if (t < w && c0 + t < C) atomicMax(&mx[c0 + t], red[t]);
      __syncthreads();
      red[t] = 0;
      __syncthreads();
    }
  } else {
    c = blockIdx.y;
    for (int64_t k = (int64_t)blockIdx.x * 256 + t; k < k1; k += (int64_t)gridDim.x * 256) up(k);
    atomicMax(&red[0], m);
    __syncthreads();
    if (t == 0) atomicMax(&mx[c], red[0]);
  }
}

// a column's grid: entries are integers of at most 54 bits times 2^-s (max < 2^E, s = 54 - E)
__device__ __forceinline__ int col_shift(u64 mx) {
  const int e = (int)(mx >> 52);  // biased exponent; 0 (zero or subnormal) as the least normal
  return 54 - (max(e, 1) - 1022);
}
// 2^-s, or a NaN where the column holds an entry that is not finite
__device__ __forceinline__ double col_quantum(u64 mx) {
  return (mx >> 52) >= 0x7FF ? NAN : scalbn(1.0, -col_shift(mx));
}

// Digit operands of one stage (128 k from word 8 (b0 + blockIdx.x)) and column group:
// dst[(group * nblk + blk) * planes * NT + plane * NT + tile][step a][1024]; lane l's 16
// bytes of a step's operand: digit column l % 16 of the tile, word 2 (l / 16) + a, byte
// 4 t + b = code slot 4 b + t.  Digit column s * Cg + c holds digit s (highest first) of the
// group's column c.  sums[2 c], [2 c + 1]: the sums of v3 on the grid, in two parts of 28
// low and the remaining high bits, so that they stay exact.
template <int KIND, int MODE>
__global__ __launch_bounds__(256) void k_cd_build(ColArgs A, int32_t layout, int64_t b0, int32_t C,
                                                  int32_t Cg, int32_t NT, const u64 *__restrict__ mx,
                                                  uint8_t *__restrict__ dst, u64 *__restrict__ sums) {
  constexpr int planes = MODE == kCdSum ? 2 : 1;
  constexpr bool rowmajor = KIND == kColPanel || KIND == kColLevB;
  __shared__ __align__(16) uint8_t img[2 * kMaxNT * 2 * kFragB];
  __shared__ u64 ssum[2 * kMaxCols];
  const int t = threadIdx.x;
  const int32_t c0 = blockIdx.y * Cg, nc = min(Cg, C - c0);
  const int64_t blk = blockIdx.x;
  const int32_t bytes = planes * NT * 2 * kFragB;
  for (int e = t * 16; e < bytes; e += 256 * 16) *(uint4 *)&img[e] = make_uint4(0, 0, 0, 0);
  if (t < 2 * kMaxCols) ssum[t] = 0;
  __syncthreads();
  for (int e = t; e < kSt * nc; e += 256) {
    const int p = rowmajor ? e / nc : e & (kSt - 1), c = rowmajor ? e % nc : e / kSt;
    const int jl = p >> 4, i = p & 15;
    const int64_t k = code_elem(layout, 8 * (b0 + blk) + jl, i);
    const u64 m = mx[c0 + c];
    if ((m >> 52) >= 0x7FF) continue;
    const int sh = col_shift(m);
    const Col3 v = col_value<KIND>(A, k, c0 + c);
    const int at = (jl & 1) * kFragB + (jl >> 1) * 256 + (i & 3) * 4 + (i >> 2);
    auto put = [&](double x, int plane) {
      int64_t q = llrint(scalbn(x, sh));
#pragma unroll
      for (int s = kDig - 1; s >= 0; --s) {
        const int32_t d = (int8_t)(q & 0xFF);
        q = (q - d) >> 8;
        const int dc = s * Cg + c;
        img[(plane * NT + (dc >> 4)) * 2 * kFragB + (dc & 15) * 16 + at] = (uint8_t)d;
      }
    };
    if (MODE == kCdMiss) {
      put(v.v2, 0);
    } else {
      put(v.v1, 0);
      if (MODE == kCdSum) put(v.v2, 1);
    }
    const int64_t q3 = llrint(scalbn(v.v3, sh));
    if (q3 != 0) {
      atomicAdd(&ssum[2 * c], (u64)(q3 & ((1 << 28) - 1)));
      atomicAdd(&ssum[2 * c + 1], (u64)(q3 >> 28));
    }
  }
  __syncthreads();
  uint8_t *out = dst + ((int64_t)blockIdx.y * gridDim.x + blk) * bytes;
  for (int e = t * 16; e < bytes; e += 256 * 16) *(uint4 *)(out + e) = *(uint4 *)&img[e];
  if (t < 2 * nc && ssum[t] != 0) atomicAdd(&sums[2 * c0 + t], ssum[t]);
}

// ------------------------------------------------------------------ the product
struct MulArgs {
  CodeView v;
  const uint8_t *dig;
  int32_t *part;      // [group][split][2 for kCdPair][rowpad][NT * 16]
  int64_t nblk;       // stages
  int64_t per;        // stages per split
  int32_t nrowblk, ngroup, nsplit;
  int64_t rowpad;
  int32_t accum;      // add to what part holds
};

// One block per (row block, split, group): four waves of R row tiles of 16.  MODE kCdPair
// multiplies one digit set with the codes and with the missing bits into two sums, kCdSum
// two sets into one, kCdMiss one set with the missing bits.  A stage's digits (NT tiles x
// planes x 2 KB) go through one of two LDS buffers, loaded into registers a stage ahead;
// the codes come straight from memory, a word pair per lane and row tile.  R = 4 (two
// for kCdPair, whose operands feed twice the products) keeps an operand read from LDS in
// use for 64 cycles of MFMA, half the LDS' rate.
template <int NT, int MODE, int R>
__global__ __launch_bounds__(256, 2) void k_cd_mul(MulArgs A) {
  constexpr int planes = MODE == kCdSum ? 2 : 1, nacc = MODE == kCdPair ? 2 : 1;
  constexpr int bytes = planes * NT * 2 * kFragB, nld = bytes / 4096;
  constexpr int tail = bytes % 4096;  // 0 or 2048: the last 128 threads' worth
  __shared__ __align__(16) uint8_t lds[2][bytes];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, q = lane >> 4;
  const int64_t item = blockIdx.x;
  const int32_t grp = (int32_t)(item % A.ngroup);
  const int32_t rb = (int32_t)((item / A.ngroup) % A.nrowblk);
  const int32_t split = (int32_t)(item / ((int64_t)A.ngroup * A.nrowblk));
  const int64_t k0 = split * A.per, k1 = min(A.nblk, k0 + A.per);
  const uint8_t *dig = A.dig + ((int64_t)grp * A.nblk) * bytes;
  const int64_t r0 = ((int64_t)rb * 4 + w) * (16 * R);
  const uint8_t *rp[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = min(r0 + 16 * r + (lane & 15), (int64_t)A.v.nrow - 1);
    const uint8_t *b = A.v.rows ? A.v.rows[row] : A.v.base + (row >> 7) * A.v.RT + (row & 127) * A.v.RS;
    rp[r] = b + (q >> 1) * A.v.QH + (q & 1) * 8;
  }
  // the word pairs past the last one read as missing (their digits are zero)
  auto codes = [&](int64_t k, uint2 (&cw)[R]) {
    const bool in = k < k1 && 8 * k + 2 * q < A.v.nword;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      cw[r] = make_uint2(~0u, ~0u);
      if (in) cw[r] = *(const uint2 *)(rp[r] + k * A.v.KB);
    }
  };
  i32x4 st[nld + 1];
  auto load = [&](int64_t k) {
    const uint8_t *s = dig + min(k, k1 - 1) * bytes + t * 16;
#pragma unroll
    for (int u = 0; u < nld; ++u) st[u] = *(const i32x4 *)(s + u * 4096);
    if (tail && t < 128) st[nld] = *(const i32x4 *)(s + nld * 4096);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < nld; ++u) *(i32x4 *)&lds[buf][t * 16 + u * 4096] = st[u];
    if (tail && t < 128) *(i32x4 *)&lds[buf][t * 16 + nld * 4096] = st[nld];
  };
  i32x4 acc[nacc][NT][R];
  int32_t *out = A.part + (((int64_t)grp * A.nsplit + split) * nacc) * A.rowpad * (NT * 16);
#pragma unroll
  for (int a = 0; a < nacc; ++a)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        acc[a][n][r] = i32x4{0, 0, 0, 0};
        if (A.accum)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[a][n][r][e] = out[(a * A.rowpad + r0 + 16 * r + 4 * q + e) * (NT * 16) + 16 * n + (lane & 15)];
      }
  uint2 cw[R], cn[R];
  load(k0);
  codes(k0, cw);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int64_t k = k0; k < k1; ++k) {
    load(k + 1);
    codes(k + 1, cn);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      i32x4 fc[R], fm[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t x = a ? cw[r].y : cw[r].x;
        const uint32_t ms = x & (x >> 1) & 0x55555555u;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          fc[r][u] = (int)((x >> (2 * u)) & 0x03030303u);
          fm[r][u] = (int)((ms >> (2 * u)) & 0x01010101u);
        }
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const i32x4 d0 = *(const i32x4 *)&lds[buf][(2 * n + a) * kFragB + lane * 16];
        if constexpr (MODE == kCdPair) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            acc[0][n][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fc[r], d0, acc[0][n][r], 0, 0, 0);
            acc[1][n][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm[r], d0, acc[1][n][r], 0, 0, 0);
          }
        } else if constexpr (MODE == kCdSum) {
          const i32x4 d1 = *(const i32x4 *)&lds[buf][(2 * (NT + n) + a) * kFragB + lane * 16];
#pragma unroll
          for (int r = 0; r < R; ++r)
            acc[0][n][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fc[r], d0, acc[0][n][r], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < R; ++r)
            acc[0][n][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm[r], d1, acc[0][n][r], 0, 0, 0);
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r)
            acc[0][n][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm[r], d0, acc[0][n][r], 0, 0, 0);
        }
      }
    }
    store(buf ^ 1);
#pragma unroll
    for (int r = 0; r < R; ++r) cw[r] = cn[r];
    __syncthreads();
    buf ^= 1;
  }
  // v_mfma_i32_16x16x64: lane l, result e holds D[4 (l / 16) + e][l % 16]
#pragma unroll
  for (int a = 0; a < nacc; ++a)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          out[(a * A.rowpad + r0 + 16 * r + 4 * q + e) * (NT * 16) + 16 * n + (lane & 15)] = acc[a][n][r][e];
}

// ------------------------------------------------------------------ results
// column j (of its group's Cg) of one row: the digits' sum over the splits, in units of
// the column's grid, as hi * 2^24 + lo, both exact
__device__ __forceinline__ void digit_sum(const int32_t *__restrict__ p, int64_t step, int32_t nsplit,
                                          int32_t Cg, int64_t &hi, int64_t &lo) {
  hi = lo = 0;
#pragma unroll
  for (int s = 0; s < kDig; ++s) {
    int64_t v = 0;
#pragma unroll 8
    for (int32_t sp = 0; sp < nsplit; ++sp) v += p[sp * step + s * Cg];
    if (s < 4) hi = hi * 256 + v;
    else lo = lo * 256 + v;
  }
}
__device__ __forceinline__ double two_parts(int64_t hi, int64_t lo) {
  return fma((double)hi, 16777216.0, (double)lo);
}

// rows = samples: total + sum of v3, all on the grid, times it and `scale`; out[row * ldr
// + c * ldc] (added to what it holds with `add`); the columns C .. Cpad - 1 are zero
__global__ __launch_bounds__(256) void k_cd_out_sum(const int32_t *__restrict__ part, int32_t NTc,
                                                    int64_t rowpad, int32_t nsplit, int32_t Cg,
                                                    int32_t C, int32_t Cpad, int64_t nrow,
                                                    const u64 *__restrict__ mx,
                                                    const u64 *__restrict__ sums, double scale,
                                                    double *__restrict__ out, int64_t ldr, int64_t ldc,
                                                    int32_t add) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = e / Cpad;
  const int32_t c = (int32_t)(e % Cpad);
  if (row >= nrow) return;
  double v = 0.0;
  if (c < C) {
    const int32_t g = c / Cg, j = c % Cg;
    const int64_t step = rowpad * NTc;
    int64_t hi, lo;
    digit_sum(part + (int64_t)g * nsplit * step + row * NTc + j, step, nsplit, Cg, hi, lo);
    // the sums' parts split at 28 bits, the digits' at 24
    const int64_t s0 = (int64_t)sums[2 * c], s1 = (int64_t)sums[2 * c + 1];
    hi += 16 * s1;
    lo += s0;
    v = two_parts(hi, lo) * col_quantum(mx[c]) * scale;
  }
  double *o = out + row * ldr + c * ldc;
  *o = add ? *o + v : v;
}

// rows = SNPs: f (C - 3 M) + l0 (S - M) times `scale`, C and M the sums over the codes and
// the missing bits, S the column's own; zero where ignore (may be null) is set
__global__ __launch_bounds__(256) void k_cd_out_pair(const int32_t *__restrict__ part, int32_t NTc,
                                                     int64_t rowpad, int32_t nsplit, int32_t Cg,
                                                     int32_t C, int64_t nrow,
                                                     const u64 *__restrict__ mx,
                                                     const u64 *__restrict__ sums,
                                                     const double *__restrict__ lev,
                                                     const uint8_t *__restrict__ ignore, double scale,
                                                     double *__restrict__ out, int64_t ldr, int64_t ldc) {
  int64_t row;
  int32_t c;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (ldc == 1) {
    row = e / C;
    c = (int32_t)(e % C);
  } else {
    row = e % nrow;
    c = (int32_t)(e / nrow);
    if (c >= C) return;
  }
  if (row >= nrow) return;
  double v = 0.0;
  if (!ignore || !ignore[row]) {
    const int32_t g = c / Cg, j = c % Cg;
    const int64_t plane = rowpad * NTc, step = 2 * plane;
    const int32_t *p = part + (int64_t)g * nsplit * step + row * NTc + j;
    int64_t ch, cl, mh, ml;
    digit_sum(p, step, nsplit, Cg, ch, cl);
    digit_sum(p + plane, step, nsplit, Cg, mh, ml);
    const double l0 = lev[4 * row], f = 0.5 * (lev[4 * row + 2] - l0);
    const double x = two_parts(ch - 3 * mh, cl - 3 * ml);
    const double y = two_parts(16 * (int64_t)sums[2 * c + 1] - mh, (int64_t)sums[2 * c] - ml);
    v = (f * x + l0 * y) * col_quantum(mx[c]) * scale;
  }
  out[row * ldr + c * ldc] = v;
}

template <int KIND, int MODE, int NT>
void launch_mul(const MulArgs &A, hipStream_t st) {
  constexpr int R = MODE == kCdPair ? 2 : 4;
  hipLaunchKernelGGL((k_cd_mul<NT, MODE, R>), dim3((unsigned)((int64_t)A.nrowblk * A.ngroup * A.nsplit)),
                     dim3(256), 0, st, A);
}
}  // namespace

// column groups: at most 20 columns (nine tiles), or 11 (five) when that is all
static void cd_groups(int32_t C, int32_t &ngroup, int32_t &Cg, int32_t &NT) {
  ngroup = (C + kMaxCols - 1) / kMaxCols;
  Cg = (C + ngroup - 1) / ngroup;
  NT = Cg * kDig <= 80 ? 5 : 9;
}

CodesPlan eig_codes_plan(const eig_ctx *ctx, int mode, int32_t C, int64_t nrow, int64_t nblk,
                         int32_t smax) {
  CodesPlan P;
  P.mode = mode;
  P.C = C;
  P.nblk = nblk;
  cd_groups(C, P.ngroup, P.Cg, P.NT);
  const int32_t rows = mode == kCdPair ? 128 : 256;
  P.nrowblk = (int32_t)((nrow + rows - 1) / rows);
  P.rowpad = (int64_t)P.nrowblk * rows;
  // splits: rounds of the blocks the chip holds (two per CU) times stages each, plus the
  // sums' way to memory and back, worth about two stages a block
  const int64_t slots = 2 * (int64_t)std::max(ctx->num_cu, 1);
  double best = 0.0;
  P.nsplit = 1;
  P.per = nblk;
  for (int32_t s = 1; s <= (int32_t)std::min<int64_t>(nblk, std::max<int64_t>(smax, nblk * kSt / kCodesMaxK + 2)); ++s) {
    const int64_t pe = (nblk + s - 1) / s;
    if ((nblk + pe - 1) / pe != s) continue;
    if (pe * kSt > kCodesMaxK) continue;  // INT32 sums
    const double rounds = (double)(((int64_t)P.nrowblk * P.ngroup * s + slots - 1) / slots);
    const double cost = rounds * ((double)pe + 2.0) + 1.0 * (double)P.nrowblk * P.ngroup * s / slots;
    if (best == 0.0 || cost < best) {
      best = cost;
      P.nsplit = s;
      P.per = pe;
    }
  }
  const int32_t planes = mode == kCdSum ? 2 : 1, nacc = mode == kCdPair ? 2 : 1;
  P.head_bytes = ((size_t)C * 24 + 255) / 256 * 256;
  P.dig_bytes = (size_t)P.ngroup * nblk * planes * P.NT * 2 * kFragB;
  P.part_bytes = (size_t)P.ngroup * P.nsplit * nacc * P.rowpad * P.NT * 16 * 4;
  return P;
}

#define CD_KIND(K, ...)              \
  case K: {                          \
    constexpr int KIND = K;          \
    __VA_ARGS__;                     \
  } break;
#define CD_KINDS(k, ...)                                                       \
  switch (k) {                                                                 \
    CD_KIND(kColPanel, __VA_ARGS__) CD_KIND(kColAxes, __VA_ARGS__)             \
    CD_KIND(kColLevB, __VA_ARGS__) CD_KIND(kColFx, __VA_ARGS__)                \
    CD_KIND(kColLsqR, __VA_ARGS__) CD_KIND(kColLsqG, __VA_ARGS__)              \
  }

static ColArgs col_args(const CodeCols &c) {
  return ColArgs{c.a, c.ld, c.n, c.lev, c.fancy, c.xmean, c.ignore, c.fxscal, c.K};
}

// column scales over all of k (head: [C] maxima, [2 C] sums), once per product
int eig_codes_scales(eig_ctx *ctx, const CodesPlan &P, const CodeCols &cols, void *head, hipStream_t st) {
  u64 *mx = (u64 *)head;
  const ColArgs A = col_args(cols);
  hipLaunchKernelGGL(k_cd_zero, dim3((unsigned)((3 * P.C + 255) / 256)), dim3(256), 0, st, mx, 3 * P.C);
  const bool rm = cols.kind == kColPanel || cols.kind == kColLevB;
  const int64_t per = rm ? std::max(1, 256 / std::min(P.C, 256)) : 256;
  const unsigned gx = (unsigned)std::min<int64_t>((cols.n + per - 1) / per, rm ? 2048 : 64);
  CD_KINDS(cols.kind, hipLaunchKernelGGL((k_cd_max<KIND>), dim3(gx, rm ? 1 : (unsigned)P.C), dim3(256), 0,
                                         st, A, cols.n, P.C, mx));
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

// the sums of v3 back to zero, for another range of k under the same scales
int eig_codes_restart(eig_ctx *ctx, const CodesPlan &P, void *head, hipStream_t st) {
  hipLaunchKernelGGL(k_cd_zero, dim3((unsigned)((2 * P.C + 255) / 256)), dim3(256), 0, st,
                     (u64 *)head + P.C, 2 * P.C);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

// digit operands of stages b0 .. b0 + P.nblk - 1 and the product of the view's codes with
// them, into part (added to it with accum)
int eig_codes_mul(eig_ctx *ctx, const CodesPlan &P, const CodeView &v, const CodeCols &cols, int64_t b0,
                  void *head, void *dig, void *part, bool accum, hipStream_t st) {
  const ColArgs A = col_args(cols);
  const u64 *mx = (const u64 *)head;
  u64 *sums = (u64 *)head + P.C;
  const dim3 grid((unsigned)P.nblk, (unsigned)P.ngroup);
  CD_KINDS(cols.kind,
           constexpr int MODE = KIND == kColPanel || KIND == kColAxes ? kCdPair
                                : KIND == kColLsqG                    ? kCdMiss
                                                                      : kCdSum;
           hipLaunchKernelGGL((k_cd_build<KIND, MODE>), grid, dim3(256), 0, st, A, v.layout, b0, P.C, P.Cg,
                              P.NT, mx, (uint8_t *)dig, sums));
  MulArgs m{v, (const uint8_t *)dig, (int32_t *)part, P.nblk, P.per, P.nrowblk, P.ngroup, P.nsplit,
            P.rowpad, accum ? 1 : 0};
  CD_KINDS(cols.kind,
           constexpr int MODE = KIND == kColPanel || KIND == kColAxes ? kCdPair
                                : KIND == kColLsqG                    ? kCdMiss
                                                                      : kCdSum;
           if (P.NT == 5) launch_mul<KIND, MODE, 5>(m, st); else launch_mul<KIND, MODE, 9>(m, st));
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

int eig_codes_out_sum(eig_ctx *ctx, const CodesPlan &P, int64_t nrow, const void *head, const void *part,
                      double scale, double *out, int64_t ldr, int64_t ldc, int32_t Cpad, bool add,
                      hipStream_t st) {
  const u64 *mx = (const u64 *)head;
  hipLaunchKernelGGL(k_cd_out_sum, dim3((unsigned)((nrow * Cpad + 255) / 256)), dim3(256), 0, st,
                     (const int32_t *)part, P.NT * 16, P.rowpad, P.nsplit, P.Cg, P.C, Cpad, nrow, mx,
                     mx + P.C, scale, out, ldr, ldc, add ? 1 : 0);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

int eig_codes_out_pair(eig_ctx *ctx, const CodesPlan &P, int64_t nrow, const void *head, const void *part,
                       const double *lev, const uint8_t *ignore, double scale, double *out, int64_t ldr,
                       int64_t ldc, hipStream_t st) {
  const u64 *mx = (const u64 *)head;
  hipLaunchKernelGGL(k_cd_out_pair, dim3((unsigned)((nrow * P.C + 255) / 256)), dim3(256), 0, st,
                     (const int32_t *)part, P.NT * 16, P.rowpad, P.nsplit, P.Cg, P.C, nrow, mx, mx + P.C,
                     lev, ignore, scale, out, ldr, ldc);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}
