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
// split.  The grid is the column's, though: where its largest entry stands far above the sum of
// the others that a row sees (and the row lacks that entry), FP64 accumulation keeps more.  With
// n entries seen, of mean size a, that is where the largest exceeds about n a.
//
// Used by fastmode's FP64 panel products (kjg_fpca.c:104-178), the SNP loadings and their
// scales (smartpca.c:1438-1525) and lsqproject's normal equations (smartpca.c:4606-4757).
#include <algorithm>
#include <cmath>

#include "eig_internal.h"

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4;
typedef unsigned long long u64;

namespace {
// ------------------------------------------------------------------ columns
// The three FP64 values of column c at index k: v1 multiplies the code, v2 = -(3 v1 + v3) the
// missing bit, v3 is summed alone.  (Columns over samples multiply both with one value.)
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
// dst[(((group * nblk + blk) * 2 + step a) * planes + plane) * NT + tile][1024]; lane l's 16
// bytes of a step's operand: digit column l % 16 of the tile, word 2 (l / 16) + a, byte
// 4 t + b = code slot 4 b + t.  Digit column s * Cg + c holds digit s (highest first) of the
// group's column c.  The missing bit's plane is formed from the other two on the grid, so
// that a missing genotype (code 3, its bit, and its share of v3's sum) adds up to zero exactly:
// v1, v2 and v3 rounded one by one left up to 2.5 steps each, 2e-13 of the right-hand side of
// a sample with 99.9 % missing.  It is within 2 steps of v2, inside the seven digits' range.
// sums[2 c], [2 c + 1]: the sums of v3 on the grid, in two parts of 28 low and the remaining
// high bits, so that they stay exact.
template <int KIND, int MODE>
__global__ __launch_bounds__(256) void k_cd_build(ColArgs A, int32_t layout, int64_t b0, int32_t C,
                                                  int32_t Cg, int32_t NT, const u64 *__restrict__ mx,
                                                  uint8_t *__restrict__ dst, u64 *__restrict__ sums) {
  constexpr int planes = MODE == kCdSum ? 2 : 1;
  constexpr bool rowmajor = KIND == kColPanel || KIND == kColLevB;
  __shared__ __align__(16) uint8_t img[2 * kCdMaxNT * 2 * kCdFrag];
  __shared__ u64 ssum[2 * kCdMaxCols];
  const int t = threadIdx.x;
  const int32_t c0 = blockIdx.y * Cg, nc = min(Cg, C - c0);
  const int64_t blk = blockIdx.x;
  const int32_t bytes = planes * NT * 2 * kCdFrag;
  for (int e = t * 16; e < bytes; e += 256 * 16) *(uint4 *)&img[e] = make_uint4(0, 0, 0, 0);
  if (t < 2 * kCdMaxCols) ssum[t] = 0;
  __syncthreads();
  // an item is one dword of an operand: the code slots u, u + 4, u + 8, u + 12 of a word
  for (int e = t; e < 32 * nc; e += 256) {
    const int p = rowmajor ? e / nc : e & 31, c = rowmajor ? e % nc : e >> 5;
    const int jl = p >> 2, u = p & 3;
    const u64 m = mx[c0 + c];
    if ((m >> 52) >= 0x7FF) continue;
    const int sh = col_shift(m);
    Col3 v[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      v[b] = col_value<KIND>(A, code_elem(layout, 8 * (b0 + blk) + jl, 4 * b + u), c0 + c);
    const int at = (jl >> 1) * 256 + u * 4;
    auto put = [&](int64_t (&q)[4], int plane) {
#pragma unroll
      for (int s = kCdDig - 1; s >= 0; --s) {
        uint32_t w = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int32_t d = (int8_t)(q[b] & 0xFF);
          q[b] = (q[b] - d) >> 8;
          w |= ((uint32_t)d & 0xFFu) << (8 * b);
        }
        const int dc = s * Cg + c;
        *(uint32_t *)&img[((jl & 1) * planes * NT + plane * NT + (dc >> 4)) * kCdFrag + (dc & 15) * 16 + at] = w;
      }
    };
    int64_t q1[4], q2[4], lo = 0, hi = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int64_t q3 = llrint(scalbn(v[b].v3, sh));
      q1[b] = llrint(scalbn(v[b].v1, sh));
      q2[b] = -(3 * q1[b] + q3);
      lo += q3 & ((1 << 28) - 1);
      hi += q3 >> 28;
    }
    if (MODE == kCdMiss) {
      put(q2, 0);
    } else {
      put(q1, 0);
      if (MODE == kCdSum) put(q2, 1);
    }
    if (lo != 0) atomicAdd(&ssum[2 * c], (u64)lo);
    if (hi != 0) atomicAdd(&ssum[2 * c + 1], (u64)hi);
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
// two sets into one, kCdMiss one set with the missing bits.  A half stage's digits (64 k:
// NT tiles x planes x 1 KB) go through one of two LDS buffers, loaded into registers half a
// stage ahead; the codes come straight from memory, a word pair per lane and row tile.
// R = 4 (two for kCdPair, whose operands feed twice the products) keeps an operand read
// from LDS in use for 64 cycles of MFMA, half the LDS' rate; nine tiles of two planes take
// R = 3, whose sums leave registers for both planes' operands (R = 4 spilled 14 to 50).
template <int NT, int MODE, int R>
__global__ __launch_bounds__(256, 2) void k_cd_mul(MulArgs A) {
  constexpr int planes = MODE == kCdSum ? 2 : 1, nacc = MODE == kCdPair ? 2 : 1;
  constexpr int bytes = planes * NT * kCdFrag, nld = bytes / 4096;  // of a half stage
  constexpr int tail = bytes % 4096 / 16;  // threads with one more piece
  __shared__ __align__(16) uint8_t lds[2][bytes];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, q = lane >> 4;
  const int64_t item = blockIdx.x;
  const int32_t grp = (int32_t)(item % A.ngroup);
  const int32_t rb = (int32_t)((item / A.ngroup) % A.nrowblk);
  const int32_t split = (int32_t)(item / ((int64_t)A.ngroup * A.nrowblk));
  const int64_t k0 = split * A.per, k1 = min(A.nblk, k0 + A.per);
  const uint8_t *dig = A.dig + ((int64_t)grp * A.nblk) * (2 * bytes) + t * 16;
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
  auto load = [&](int64_t h) {  // half stage h, or the last one again past the end
    const uint8_t *s = dig + min(h, 2 * k1 - 1) * bytes;
#pragma unroll
    for (int u = 0; u < nld; ++u) st[u] = *(const i32x4 *)(s + u * 4096);
    if (tail && t < tail) st[nld] = *(const i32x4 *)(s + nld * 4096);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < nld; ++u) *(i32x4 *)&lds[buf][t * 16 + u * 4096] = st[u];
    if (tail && t < tail) *(i32x4 *)&lds[buf][t * 16 + nld * 4096] = st[nld];
  };
  i32x4 acc[nacc][NT][R];
#pragma unroll
  for (int a = 0; a < nacc; ++a)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[a][n][r] = i32x4{0, 0, 0, 0};
  uint2 cw[R], cn[R];
  load(2 * k0);
  codes(k0, cw);
  store(0);
  __syncthreads();
  for (int64_t k = k0; k < k1; ++k) {
    codes(k + 1, cn);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      load(2 * k + a + 1);
      auto code_op = [&](i32x4 (&f)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const uint32_t x = a ? cw[r].y : cw[r].x;
#pragma unroll
          for (int u = 0; u < 4; ++u) f[r][u] = (int)((x >> (2 * u)) & 0x03030303u);
        }
      };
      auto miss_op = [&](i32x4 (&f)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const uint32_t x = a ? cw[r].y : cw[r].x, ms = x & (x >> 1) & 0x55555555u;
#pragma unroll
          for (int u = 0; u < 4; ++u) f[r][u] = (int)((ms >> (2 * u)) & 0x01010101u);
        }
      };
      auto dig_op = [&](int n) { return *(const i32x4 *)&lds[a][n * kCdFrag + lane * 16]; };
      auto mul = [&](const i32x4 (&f)[R], const i32x4 &d, i32x4 (&c)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) c[r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[r], d, c[r], 0, 0, 0);
      };
      i32x4 fc[R], fm[R];
      if constexpr (MODE != kCdMiss) code_op(fc);
      miss_op(fm);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const i32x4 d = dig_op(n);
        if constexpr (MODE == kCdPair) {
          mul(fc, d, acc[0][n]);
          mul(fm, d, acc[nacc - 1][n]);
        } else if constexpr (MODE == kCdSum) {
          mul(fc, d, acc[0][n]);
          mul(fm, dig_op(NT + n), acc[0][n]);
        } else {
          mul(fm, d, acc[0][n]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      store(a ^ 1);
      __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) cw[r] = cn[r];
  }
  // v_mfma_i32_16x16x64: lane l, result e holds D[4 (l / 16) + e][l % 16]
  int32_t *out = A.part + (((int64_t)grp * A.nsplit + split) * nacc) * A.rowpad * (NT * 16) +
                 (r0 + 4 * q) * (NT * 16) + (lane & 15);
  const bool more = A.accum != 0;
#pragma unroll 1
  for (int a = 0; a < nacc; ++a) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          int32_t *o = out + (16 * r + e) * (NT * 16) + 16 * n;
          const int v = nacc == 2 && a == 1 ? acc[nacc - 1][n][r][e] : acc[0][n][r][e];
          *o = more ? *o + v : v;
        }
    out += A.rowpad * (NT * 16);
  }
}

// ---- up to 16 rows: one row tile, so the digits are read once and bound the product.
// A wave streams the digit operands of its range of stages straight from memory, a half
// stage (NT x planes KB) ahead of its MFMAs; nothing is shared between waves.
// part[grp][split][row < nrow][NT * 16].
template <int NT, int MODE>
__global__ __launch_bounds__(256) void k_cd_stream(const uint8_t *__restrict__ dig_, int32_t *__restrict__ part,
                                                   CodeRows rows, int64_t nword, int64_t nblk, int64_t per,
                                                   int32_t ngroup, int32_t nsplit) {
  constexpr int planes = MODE == kCdSum ? 2 : 1, F = planes * NT, bytes = F * kCdFrag;
  const int lane = threadIdx.x & 63, q = lane >> 4;
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= (int64_t)ngroup * nsplit) return;
  const int32_t grp = (int32_t)(item % ngroup), split = (int32_t)(item / ngroup);
  const int64_t k0 = split * per, k1 = min(nblk, k0 + per);
  const uint8_t *rp = rows.row[min(lane & 15, rows.n - 1)] + q * 8;
  const uint8_t *dig = dig_ + (grp * nblk) * (2 * bytes) + lane * 16;
  i32x4 acc[NT], f[F], g[F];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = i32x4{0, 0, 0, 0};
  auto load = [&](int64_t h, i32x4 (&d)[F]) {
    const uint8_t *s = dig + min(h, 2 * k1 - 1) * bytes;
#pragma unroll
    for (int n = 0; n < F; ++n) d[n] = *(const i32x4 *)(s + n * kCdFrag);
  };
  auto codes = [&](int64_t k) {
    uint2 c = make_uint2(~0u, ~0u);
    if (k < k1 && 8 * k + 2 * q < nword) c = *(const uint2 *)(rp + k * 32);
    return c;
  };
  auto mul = [&](uint32_t x, const i32x4 (&d)[F]) {
    const uint32_t ms = x & (x >> 1) & 0x55555555u;
    i32x4 fc, fm;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      fc[u] = (int)((x >> (2 * u)) & 0x03030303u);
      fm[u] = (int)((ms >> (2 * u)) & 0x01010101u);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      if (MODE == kCdSum) acc[n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fc, d[n], acc[n], 0, 0, 0);
      acc[n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm, d[(planes - 1) * NT + n], acc[n], 0, 0, 0);
    }
  };
  load(2 * k0, f);
  uint2 cw = codes(k0);
  for (int64_t k = k0; k < k1; ++k) {
    load(2 * k + 1, g);
    const uint2 cn = codes(k + 1);
    mul(cw.x, f);
    load(2 * k + 2, f);
    mul(cw.y, g);
    cw = cn;
  }
  int32_t *out = part + ((int64_t)grp * nsplit + split) * rows.n * (NT * 16) + (lane & 15);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (4 * q + e < rows.n)
#pragma unroll
      for (int n = 0; n < NT; ++n) out[(4 * q + e) * (NT * 16) + 16 * n] = acc[n][e];
}

// ------------------------------------------------------------------ results
// kOutRows rows of one group's sums, over the splits, in LDS: a block reads them in whole
// lines (a thread per result reading its digits from memory took 1.3 ms for 600,000 rows
// of ten columns stored by column, now 0.19, and 0.13 for 100,000 of twenty, now 0.10)
constexpr int kOutRows = 16;
template <int NACC>
__device__ __forceinline__ void out_rows(const int32_t *__restrict__ part, int32_t NTc, int64_t rowpad,
                                         int32_t nsplit, int64_t row0, int64_t *sm) {
  const int64_t plane = rowpad * NTc;
#pragma unroll
  for (int a = 0; a < NACC; ++a) {
    const int32_t *p = part + a * plane + row0 * NTc;
    for (int e = threadIdx.x * 4; e < kOutRows * NTc; e += 1024) {
      int64_t v[4] = {0, 0, 0, 0};
#pragma unroll 4
      for (int32_t sp = 0; sp < nsplit; ++sp) {
        const i32x4 x = *(const i32x4 *)(p + sp * (NACC * plane) + e);
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] += x[u];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) sm[a * kOutRows * NTc + e + u] = v[u];
    }
  }
  __syncthreads();
}
// a column's digits in units of its grid, as hi * 2^24 + lo, both exact
__device__ __forceinline__ void digit_sum(const int64_t *p, int32_t Cg, int64_t &hi, int64_t &lo) {
  hi = lo = 0;
#pragma unroll
  for (int s = 0; s < kCdDig; ++s) {
    if (s < 4) hi = hi * 256 + p[s * Cg];
    else lo = lo * 256 + p[s * Cg];
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
  __shared__ int64_t sm[kOutRows * kCdMaxNT * 16];
  const int64_t row0 = (int64_t)blockIdx.x * kOutRows;
  const int32_t g = blockIdx.y, c0 = g * Cg, c1 = g + 1 == (int32_t)gridDim.y ? Cpad : c0 + Cg;
  out_rows<1>(part + (int64_t)g * nsplit * rowpad * NTc, NTc, rowpad, nsplit, row0, sm);
  const int32_t w = c1 - c0;
  for (int e = threadIdx.x; e < kOutRows * w; e += 256) {
    const int r = ldc == 1 ? e / w : e % kOutRows, j = ldc == 1 ? e % w : e / kOutRows;
    const int64_t row = row0 + r;
    const int32_t c = c0 + j;
    if (row >= nrow) continue;
    double v = 0.0;
    if (c < C) {
      int64_t hi, lo;
      digit_sum(sm + r * NTc + j, Cg, hi, lo);
      // the sums' parts split at 28 bits, the digits' at 24
      hi += 16 * (int64_t)sums[2 * c + 1];
      lo += (int64_t)sums[2 * c];
      v = two_parts(hi, lo) * col_quantum(mx[c]) * scale;
    }
    double *o = out + row * ldr + c * ldc;
    *o = add ? *o + v : v;
  }
}

// The results of kCdSum and kCdMiss over many splits: one block per (row, group), seven
// slices of the splits side by side (part[grp][split][rowpad][NTc])
__global__ __launch_bounds__(1024) void k_cd_out_small(const int32_t *__restrict__ part, int32_t NTc,
                                                       int64_t rowpad, int32_t nsplit, int32_t Cg, int32_t C,
                                                       const u64 *__restrict__ mx,
                                                       const u64 *__restrict__ sums,
                                                       double *__restrict__ out, int64_t ldr) {
  __shared__ int64_t sl[7][kCdMaxNT * 16], sm[kCdMaxNT * 16];
  const int32_t row = blockIdx.x, g = blockIdx.y;
  const int t = threadIdx.x, j = t % NTc, s = t / NTc;
  if (s < 7) {
    int64_t v = 0;
    const int32_t *p = part + ((int64_t)g * nsplit * rowpad + row) * NTc + j;
#pragma unroll 8
    for (int32_t sp = s; sp < nsplit; sp += 7) v += p[sp * rowpad * NTc];
    sl[s][j] = v;
  }
  __syncthreads();
  if (t < NTc) {
    int64_t v = 0;
#pragma unroll
    for (int u = 0; u < 7; ++u) v += sl[u][t];
    sm[t] = v;
  }
  __syncthreads();
  const int32_t c = g * Cg + t;
  if (t < Cg && c < C) {
    int64_t hi, lo;
    digit_sum(sm + t, Cg, hi, lo);
    out[row * ldr + c] = two_parts(hi + 16 * (int64_t)sums[2 * c + 1], lo + (int64_t)sums[2 * c]) *
                         col_quantum(mx[c]);
  }
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
  __shared__ int64_t sm[2 * kOutRows * kCdMaxNT * 16];
  const int64_t row0 = (int64_t)blockIdx.x * kOutRows;
  const int32_t g = blockIdx.y, c0 = g * Cg, w = min(Cg, C - c0);
  out_rows<2>(part + (int64_t)g * nsplit * 2 * rowpad * NTc, NTc, rowpad, nsplit, row0, sm);
  for (int e = threadIdx.x; e < kOutRows * w; e += 256) {
    const int r = ldc == 1 ? e / w : e % kOutRows, j = ldc == 1 ? e % w : e / kOutRows;
    const int64_t row = row0 + r;
    const int32_t c = c0 + j;
    if (row >= nrow) continue;
    double v = 0.0;
    if (!ignore || !ignore[row]) {
      int64_t ch, cl, mh, ml;
      digit_sum(sm + r * NTc + j, Cg, ch, cl);
      digit_sum(sm + (kOutRows + r) * NTc + j, Cg, mh, ml);
      const double l0 = lev[4 * row], f = 0.5 * (lev[4 * row + 2] - l0);
      const double x = two_parts(ch - 3 * mh, cl - 3 * ml);
      const double y = two_parts(16 * (int64_t)sums[2 * c + 1] - mh, (int64_t)sums[2 * c] - ml);
      v = (f * x + l0 * y) * col_quantum(mx[c]) * scale;
    }
    out[row * ldr + c * ldc] = v;
  }
}

template <int MODE, int NT>
void launch_mul(const MulArgs &A, int R, hipStream_t st) {
  constexpr int RX = cd_tiles(MODE, NT);
  const dim3 grid((unsigned)((int64_t)A.nrowblk * A.ngroup * A.nsplit));
  if (R == 1) hipLaunchKernelGGL((k_cd_mul<NT, MODE, 1>), grid, dim3(256), 0, st, A);
  else if (R == 2) hipLaunchKernelGGL((k_cd_mul<NT, MODE, 2>), grid, dim3(256), 0, st, A);
  else hipLaunchKernelGGL((k_cd_mul<NT, MODE, RX>), grid, dim3(256), 0, st, A);
}
}  // namespace

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

// digit operands of stages b0 .. b0 + P.nblk - 1 (and the sums of v3 there, added to head's)
int eig_codes_build(eig_ctx *ctx, const CodesPlan &P, const CodeCols &cols, int32_t layout, int64_t b0,
                    void *head, void *dig, hipStream_t st) {
  const ColArgs A = col_args(cols);
  const u64 *mx = (const u64 *)head;
  u64 *sums = (u64 *)head + P.C;
  const dim3 grid((unsigned)P.nblk, (unsigned)P.ngroup);
  CD_KINDS(cols.kind,
           constexpr int MODE = KIND == kColPanel || KIND == kColAxes ? kCdPair
                                : KIND == kColLsqG                    ? kCdMiss
                                                                      : kCdSum;
           hipLaunchKernelGGL((k_cd_build<KIND, MODE>), grid, dim3(256), 0, st, A, layout, b0, P.C, P.Cg,
                              P.NT, mx, (uint8_t *)dig, sums));
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

// the product of the view's codes with P.nblk stages of digits, into part (added to it
// with accum)
hipError_t eig_codes_product(const CodesPlan &P, const CodeView &v, const void *dig, void *part,
                             bool accum, hipStream_t st) {
  MulArgs m{v, (const uint8_t *)dig, (int32_t *)part, P.nblk, P.per, P.nrowblk, P.ngroup, P.nsplit,
            P.rowpad, accum ? 1 : 0};
  if (P.mode == kCdPair) {
    if (P.NT == 5) launch_mul<kCdPair, 5>(m, P.R, st); else launch_mul<kCdPair, 9>(m, P.R, st);
  } else if (P.mode == kCdSum) {
    if (P.NT == 5) launch_mul<kCdSum, 5>(m, P.R, st); else launch_mul<kCdSum, 9>(m, P.R, st);
  } else {
    if (P.NT == 5) launch_mul<kCdMiss, 5>(m, P.R, st); else launch_mul<kCdMiss, 9>(m, P.R, st);
  }
  return hipGetLastError();
}

int eig_codes_mul(eig_ctx *ctx, const CodesPlan &P, const CodeView &v, const CodeCols &cols, int64_t b0,
                  void *head, void *dig, void *part, bool accum, hipStream_t st) {
  EIG_TRY(eig_codes_build(ctx, P, cols, v.layout, b0, head, dig, st));
  EIG_HIP(ctx, eig_codes_product(P, v, dig, part, accum, st));
  return EIG_OK;
}

hipError_t eig_codes_sum(const CodesPlan &P, int64_t nrow, const void *head, const void *part, double scale,
                         double *out, int64_t ldr, int64_t ldc, int32_t Cpad, bool add, hipStream_t st) {
  const u64 *mx = (const u64 *)head;
  // a block per row where the splits are many: 16 rows a block add them one after another
  if (P.nsplit > 8 && nrow <= 4096 && ldc == 1 && Cpad == P.C && scale == 1.0 && !add) {
    hipLaunchKernelGGL(k_cd_out_small, dim3((unsigned)nrow, (unsigned)P.ngroup), dim3(1024), 0, st,
                       (const int32_t *)part, P.NT * 16, P.rowpad, P.nsplit, P.Cg, P.C, mx, mx + P.C, out,
                       ldr);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_cd_out_sum, dim3((unsigned)((nrow + kOutRows - 1) / kOutRows), (unsigned)P.ngroup),
                     dim3(256), 0, st, (const int32_t *)part, P.NT * 16, P.rowpad, P.nsplit, P.Cg, P.C,
                     Cpad, nrow, mx, mx + P.C, scale, out, ldr, ldc, add ? 1 : 0);
  return hipGetLastError();
}

int eig_codes_out_sum(eig_ctx *ctx, const CodesPlan &P, int64_t nrow, const void *head, const void *part,
                      double scale, double *out, int64_t ldr, int64_t ldc, int32_t Cpad, bool add,
                      hipStream_t st) {
  EIG_HIP(ctx, eig_codes_sum(P, nrow, head, part, scale, out, ldr, ldc, Cpad, add, st));
  return EIG_OK;
}

// The selection's samples times cols, over all SNPs, in a workspace of eig_codes_area(P): P is
// a plan of kCdSum for all of their rows and the stages of a pass (all, or as many as its
// digits may take).  The codes come from the regrouped ones that the context keeps or, without
// them, from a range of them at a time.  The INT32 sums go on from pass to pass as long as they
// hold (their bound in SNPs), so the results are the same bits up to there.
int eig_codes_samples(eig_ctx *ctx, const CodesPlan &P, const CodeCols &cols, char *ws, int64_t nrow,
                      double scale, double *out, int64_t ldr, int64_t ldc, int32_t Cpad, hipStream_t st) {
  const int64_t rows = (int64_t)ctx->nst * kTileS, G64 = (ctx->nsnp + kGrp - 1) / kGrp, nblk = (G64 + 1) / 2;
  const bool kept = ctx->have_selg;
  const int64_t most = cd_max_k(kCdSum) / kCdStage;
  CodesPlan C = P;
  if (!kept) {
    const int64_t nb = std::min(P.nblk, eig_codes_chunk(ctx->nst, nblk));
    C = eig_codes_plan(ctx->num_cu, kCdSum, P.C, rows, nb, P.nsplit);
    EIG_TRY(eig_ensure(ctx, ctx->selg, (size_t)rows * nb * 32));
    if (eig_codes_area(C) > eig_codes_area(P)) return eig_set_err(ctx, EIG_E_STATE, "code products: work area");
  }
  char *dig = ws + C.head_bytes, *part = dig + C.dig_bytes;
  EIG_TRY(eig_codes_scales(ctx, C, cols, ws, st));
  int64_t held = 0;  // stages in an INT32 sum
  bool add = false;
  for (int64_t b0 = 0; b0 < nblk; b0 += C.nblk) {
    if (held > 0 && held + C.per > most) {
      EIG_TRY(eig_codes_out_sum(ctx, C, nrow, ws, part, scale, out, ldr, ldc, Cpad, add, st));
      EIG_TRY(eig_codes_restart(ctx, C, ws, st));
      add = true;
      held = 0;
    }
    CodeView v{(const uint8_t *)ctx->selg.p, nullptr, C.nblk * 4096, 16, 4096, 2048, rows, C.nblk * 8, kCodeGrouped};
    if (kept) {
      v.base += b0 * 4096;
      v.RT = G64 * 2048;
      v.nword = (G64 - 2 * b0) * 4;
    } else {
      EIG_TRY(eig_regroup(ctx, 2 * b0, 2 * C.nblk));
    }
    EIG_TRY(eig_codes_mul(ctx, C, v, cols, b0, ws, dig, part, held > 0, st));
    held += C.per;
  }
  return eig_codes_out_sum(ctx, C, nrow, ws, part, scale, out, ldr, ldc, Cpad, add, st);
}

int eig_codes_out_pair(eig_ctx *ctx, const CodesPlan &P, int64_t nrow, const void *head, const void *part,
                       const double *lev, const uint8_t *ignore, double scale, double *out, int64_t ldr,
                       int64_t ldc, hipStream_t st) {
  const u64 *mx = (const u64 *)head;
  hipLaunchKernelGGL(k_cd_out_pair, dim3((unsigned)((nrow + kOutRows - 1) / kOutRows), (unsigned)P.ngroup),
                     dim3(256), 0, st,
                     (const int32_t *)part, P.NT * 16, P.rowpad, P.nsplit, P.Cg, P.C, nrow, mx, mx + P.C,
                     lev, ignore, scale, out, ldr, ldc);
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

// the product of up to 16 rows (kCodeBytes layout, nword words each) and its results in
// one go: out[row * ldr + c]; kCdSum and kCdMiss.  part: eig_codes_small_bytes(P).
constexpr int32_t kSmallSplits = 512;  // waves per group: ten stages each at 600,000 SNPs
size_t eig_codes_small_bytes(const CodesPlan &P) {
  return (size_t)P.ngroup * kSmallSplits * 16 * P.NT * 16 * 4;
}
hipError_t eig_codes_small(const CodesPlan &P, const CodeRows &rows, int64_t nword, const void *head,
                           const void *dig, void *part, double *out, int64_t ldr, hipStream_t st) {
  const u64 *mx = (const u64 *)head;
  int64_t per = (P.nblk + kSmallSplits - 1) / kSmallSplits;
  const int32_t ns = (int32_t)((P.nblk + per - 1) / per);
  const dim3 grid((unsigned)(((int64_t)P.ngroup * ns + 3) / 4));
  const uint8_t *d = (const uint8_t *)dig;
  int32_t *p = (int32_t *)part;
  if (P.mode == kCdSum) {
    if (P.NT == 5) hipLaunchKernelGGL((k_cd_stream<5, kCdSum>), grid, dim3(256), 0, st, d, p, rows, nword, P.nblk, per, P.ngroup, ns);
    else hipLaunchKernelGGL((k_cd_stream<9, kCdSum>), grid, dim3(256), 0, st, d, p, rows, nword, P.nblk, per, P.ngroup, ns);
  } else {
    if (P.NT == 5) hipLaunchKernelGGL((k_cd_stream<5, kCdMiss>), grid, dim3(256), 0, st, d, p, rows, nword, P.nblk, per, P.ngroup, ns);
    else hipLaunchKernelGGL((k_cd_stream<9, kCdMiss>), grid, dim3(256), 0, st, d, p, rows, nword, P.nblk, per, P.ngroup, ns);
  }
  hipLaunchKernelGGL(k_cd_out_small, dim3((unsigned)rows.n, (unsigned)P.ngroup), dim3(1024), 0, st,
                     (const int32_t *)part, P.NT * 16, (int64_t)rows.n, ns, P.Cg, P.C, mx, mx + P.C, out, ldr);
  return hipGetLastError();
}
