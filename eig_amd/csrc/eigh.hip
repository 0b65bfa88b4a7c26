// FP64 symmetric eigensolver on the device.
//
//  1. Householder tridiagonalisation, blocked by panels of kNB columns (the
//     dsytrd/dlatrd scheme).  The working matrix is row-major and symmetric with
//     a padded leading dimension, so "column c below the diagonal" is row c right
//     of the diagonal and every access is a contiguous 16-byte pair.  Each column c
//     (panel position j) runs in two parts:
//       symv : the reflector scalars of column c (dlarfg), then y = A_trail v
//              from the upper triangle, with v rebuilt on the fly from the
//              unscaled column x; per-tile shares of y and of y.v;
//       wcol : w = tau (y - V q - W p) + alpha v, where alpha = -tau/2 w.v is
//              known up front from w.v = tau (y.v - 2 p.q); in the same pass the
//              next row x = A[c+1] - (V W^T + W V^T)[c+1] and per-block partials
//              of its norm and of the next column's panel dots V^T x, W^T x.
//     Both are launches of their own (k_symv, k_wcol).  Once the trailing matrix fits the
//     register files (order 2,048) one resident launch per range of orders runs all its
//     columns (k_tri).
//     Cross-block sums are per-block partials reduced in a fixed order (same
//     bits in every block, independent of scheduling).  After each panel
//     k_syr2k applies A -= V W^T + W V^T to the trailing matrix.  The reflector of
//     row c is left in A[c][c+1:], with tau[c].
//  2. All eigenvalues of the tridiagonal T: Sturm counts on a shared grid of the
//     Gershgorin interval, then multisection (8 to 64 lanes per eigenvalue, one
//     count each).
//  3. The top nvec eigenvectors of T by inverse iteration (LU with partial
//     pivoting, a block per vector), Gram-Schmidt inside clusters of close eigenvalues.
//  4. Back-transform X = Q Y in compact-WY form Q_p = I - V_p T_p V_p^T, last
//     panel first; all T_p are formed up front (the Gram matrices V_p^T V_p over
//     row ranges, then T_p per panel), then per panel one kernel applies the
//     previous panel and writes per-block dots V_p^T X, and a kernel with one block
//     per vector sums them in block order into Z_p = T_p V_p^T X.
//  Wave-level sums exchange lanes by DPP and permlane swaps (xlane), not through LDS.
#include <cmath>
#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "eig_internal.h"

constexpr int kNB = 32;      // panel width
constexpr int kMaxVec = 64;  // max eigenvectors computed

enum {
  S_GL = 0, S_GU, S_PIVMIN, S_TNORM, S_SCALE,
  S_COUNT
};

struct EigWs {
  double *a;  // n x lda working matrix (destroyed); columns n..lda are zero
  int32_t lda;
  double *d, *e, *e2, *tau;
  double *V, *W;  // n x kNB panel vectors (row-major)
  double *xtmp;   // current reflector column, unscaled (length lda, zero padded)
  double *yp;     // [tile][lda] shares of y = A v (k_symv)
  double *sc;
  double *part1;          // per-block partial dots of the back-transform
  double *pw;             // [2][maxw][kPW] column hand-off partials (by column parity)
  double *ps;             // per-block y.v of k_symv
  int32_t *sync;          // [1] set if a resident launch gave up waiting
  int32_t maxw;
  double *eval;           // ascending
  double2 *st;            // (d, e^2) of T scaled to a norm of 1/2 .. 1, for the Sturm counts
  double *X;              // nvec x n eigenvectors
  double *lu;             // n x 5 x kMaxVec LU factors of inverse iteration
  double *Z;              // kNB x kMaxVec
  double *Tall;           // panels x kNB x kNB
};

// Exchange of a double with lane (lane ^ o) of the wave, for o a power of two below 64
// that is a constant once the caller's loop is unrolled, without the LDS crossbar of
// ds_bpermute: o = 1, 2 and 8 by one DPP move (quad permutes; a rotation by 8 within a
// 16-lane row), o = 4 by two DPP moves (row shifts by 4 either way) and a select, o = 16
// and 32 by v_permlane16_swap / v_permlane32_swap of the value with itself and a
// select.  The values moved are those of __shfl_xor(v, o), so every sum keeps its bits.
__device__ __forceinline__ int xlane32(int v, int o) {
  const int lane = threadIdx.x & 63;
  switch (o) {
    case 1: return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);   // quad_perm 1,0,3,2
    case 2: return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);   // quad_perm 2,3,0,1
    case 4: {
      const int dn = __builtin_amdgcn_mov_dpp(v, 0x114, 0xF, 0xF, false);  // row_shr:4
      const int up = __builtin_amdgcn_mov_dpp(v, 0x104, 0xF, 0xF, false);  // row_shl:4
      return (lane & 4) ? dn : up;
    }
    case 8: return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, false);  // row_ror:8
    case 16: {  // rows 1, 3 of the first operand swap with rows 0, 2 of the second
      const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
      return (int)((lane & 16) ? r[0] : r[1]);
    }
    default: {  // lanes 32-63 of the first operand swap with lanes 0-31 of the second
      const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
      return (int)((lane & 32) ? r[0] : r[1]);
    }
  }
}
__device__ __forceinline__ double xlane(double v, int o) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)xlane32((int)(uint32_t)u, o);
  const uint32_t hi = (uint32_t)xlane32((int)(uint32_t)(u >> 32), o);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// lane 0's value in every lane (all lanes of the wave active)
__device__ __forceinline__ double lane0(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// sum over a 256-thread block; result valid in every thread.  The wave sums are trees
// over lane ^ o (lane 0 receives from lane o at each level, as with a shift down)
__device__ inline double block_sum(double v, double *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += xlane(v, o);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// ---- partials handed from part to part -------------------------------------
// Every cross-block sum is written as per-block partials and reduced, in block
// order, by the blocks of the next part:
//   wcol(c-1) -> pw[c & 1][b][kPW]: sum x^2 over rows >= c+2, x_{c+1} (alpha,
//                from block 0 only), and for q below column c's panel position
//                sum_{r >= c+2} V_q[r] x_r and sum W_q[r] x_r;
//   symv(c)   -> ps[b]: sum over its rows of y_r v_r.
constexpr int kPW = 2 + 2 * kNB;

// sum_{b = start, start+step, ... < end} p[b * stride], in that order, with the
// loads issued eight at a time so that their latencies overlap.  The first eight
// (load8) are straight-line and unconditional (indices past the end read entry
// end-1 and are discarded), so a caller can issue them together with its other
// loads and add them up later (sum_rest).  Needs start >= 0 and end >= 1.
__device__ inline void load8(const double *__restrict__ p, int64_t stride, int32_t start,
                             int32_t step, int32_t end, double (&v)[8]) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int32_t bb = start + u * step;
    const double x = p[(int64_t)min(bb, end - 1) * stride];
    v[u] = bb < end ? x : 0.0;
  }
}
__device__ __forceinline__ double sum8(const double (&v)[8]) {  // pairwise
  return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
}
__device__ inline double sum_rest(const double *__restrict__ p, int64_t stride, int32_t start,
                                  int32_t step, int32_t end, const double (&v0)[8]) {
  double s = sum8(v0);
  for (int32_t b = start + 8 * step; b < end; b += 8 * step) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int32_t bb = b + u * step;
      v[u] = bb < end ? p[(int64_t)bb * stride] : 0.0;
    }
    s += sum8(v);
  }
  return s;
}
__device__ inline double sum_strided(const double *__restrict__ p, int64_t stride, int32_t start,
                                     int32_t step, int32_t end) {
  if (end <= 0) return 0.0;
  double v[8];
  load8(p, stride, start, step, end, v);
  return sum_rest(p, stride, start, step, end, v);
}

constexpr int kWRows = 64;  // rows per w-column block (four threads per row)
__device__ inline int32_t wcol_blocks(int32_t n, int32_t c) {  // producer blocks of column c
  return c == 0 ? 1 : (n - c + kWRows - 1) / kWRows;
}

// dlarfg scalars of column c from the producers' partials, reduced by one wave in
// a fixed order (the same bits in every wave that calls it).  col_scalars_sums
// takes each lane's strided sums of the partials (sum over b = lane, lane+64, ...
// of pw[b][0] and pw[b][1]).
__device__ inline void col_scalars_sums(double s0, double s1, double &tau, double &scale,
                                        double &beta) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s0 += xlane(s0, o);
    s1 += xlane(s1, o);
  }
  s0 = lane0(s0);
  s1 = lane0(s1);
  const double alpha = s1, xn2 = s0;
  tau = 0.0;
  scale = 0.0;
  beta = alpha;
  if (xn2 > 0.0) {
    beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
    tau = (beta - alpha) / beta;
    scale = 1.0 / (alpha - beta);
  }
}
__device__ inline void col_scalars(const EigWs &ws, int32_t n, int32_t c, double &tau,
                                   double &scale, double &beta) {
  const double *pw = ws.pw + (int64_t)(c & 1) * ws.maxw * kPW;
  const int32_t nw = wcol_blocks(n, c);
  const int lane = threadIdx.x & 63;
  col_scalars_sums(sum_strided(pw, kPW, lane, 64, nw), sum_strided(pw + 1, kPW, lane, 64, nw),
                   tau, scale, beta);
}

// column 0: x = row 0, d[0], and the partials of column 0 (one block)
__global__ __launch_bounds__(256) void k_col0(EigWs ws, int32_t n) {
  __shared__ double red[4];
  double s = 0.0;
  for (int32_t r = threadIdx.x; r < n; r += 256) {
    const double x = ws.a[r];
    ws.xtmp[r] = x;
    if (r >= 2) s += x * x;
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) {
    ws.d[0] = ws.a[0];
    ws.pw[0] = s;
    ws.pw[1] = n > 1 ? ws.a[1] : 0.0;
  }
}

// one of a pair of values by a lane bit, plus the other lane's other: a step of the
// butterflies that transpose and sum.  Values, not elements of an array: a select between
// array elements becomes one of their indices
__device__ __forceinline__ double xpick(bool b, double x, double y, int o) {
  return (b ? y : x) + xlane(b ? x : y, o);
}
// tile i of the upper triangle of an nt x nt grid, counted from the last row of tiles up:
// the numbers of the tiles that are left stay the same as leading rows drop out
__device__ __forceinline__ void upper_tile(int32_t i, int32_t nt, int32_t &I, int32_t &J) {
  int32_t k = (int32_t)((sqrtf(8.0f * (float)i + 1.0f) - 1.0f) * 0.5f);
  while ((k + 1) * (k + 2) / 2 <= i) ++k;
  while (k * (k + 1) / 2 > i) --k;
  I = nt - 1 - k;
  J = I + (i - k * (k + 1) / 2);
}

// ---------------------------------------------------------------- k_symv
// y = A v from the upper triangle alone, one block per kSyT x kSyT tile of a fixed grid:
// tile (I, J) gives rows I their share of A v and, off the diagonal, rows J theirs of
// A^T v.  Row r's shares stand at yp[K][r] for the tiles K = c+1's .. nt-1 that hold it
// with its own, and k_wcol adds them in that order.  Bound by reading the triangle (from
// the Infinity Cache: 6.5 TB/s); a pass over whole rows reads twice as much.  A wave takes
// 32 rows by 128 columns, one 1 KB load per row, eight rows in flight while eight are
// summed.  A tile keeps its number from column to column, and so its XCD.
constexpr int kSyT = 128;
__host__ __device__ inline int32_t symv_tiles(int32_t n, int32_t c) {
  const int32_t k = (n + kSyT - 1) / kSyT - (c + 1) / kSyT;
  return k * (k + 1) / 2;
}
template <bool kDiag>
__device__ __forceinline__ double symv_rows8(const double2 (&a)[8], const double *sv, int32_t row,
                                             int32_t col, double v0, double v1, double &c0,
                                             double &c1) {
  double p[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const double vr = sv[u];
    double x = a[u].x, y = a[u].y, xc = x, yc = y;
    if constexpr (kDiag) {  // the tile's own upper triangle; its diagonal counts once
      x = col >= row + u ? x : 0.0;
      y = col + 1 >= row + u ? y : 0.0;
      xc = col > row + u ? x : 0.0;
      yc = col + 1 > row + u ? y : 0.0;
    }
    p[u] = fma(x, v0, y * v1);
    c0 = fma(xc, vr, c0);
    c1 = fma(yc, vr, c1);
  }
  // lane l: row l % 8 over its group of eight lanes
  const int lane = threadIdx.x & 63;
  const bool b4 = (lane & 4) != 0, b2 = (lane & 2) != 0, b1 = (lane & 1) != 0;
  const double q0 = xpick(b4, p[0], p[4], 4), q1 = xpick(b4, p[1], p[5], 4),
               q2 = xpick(b4, p[2], p[6], 4), q3 = xpick(b4, p[3], p[7], 4);
  return xpick(b1, xpick(b2, q0, q2, 2), xpick(b2, q1, q3, 2), 1);
}
__global__ __launch_bounds__(256, 4) void k_symv(EigWs ws, int32_t n, int32_t c, int32_t j) {
  __shared__ __align__(16) double sv[2 * kSyT];  // v at the tile's rows, at its columns
  __shared__ double srow[kSyT], scol[4][kSyT], red[4];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int32_t lda = ws.lda, nt = (n + kSyT - 1) / kSyT;
  int32_t I, J;
  upper_tile((int32_t)blockIdx.x, nt, I, J);
  const bool diag = I == J;
  // rows up to column c hold reflectors and rows past n nothing: they read a live row, and
  // meet v = 0 or are not stored; columns past the padding read the row's last pair
  const int32_t row = I * kSyT + 32 * wv, col = J * kSyT + 2 * lane;
  const double *ac = ws.a + min(col, lda - 2);
  double2 a[2][8];
  auto load = [&](double2 (&d)[8], int32_t r) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
      d[u] = *(const double2 *)(ac + (int64_t)min(max(r + u, c + 1), n - 1) * lda);
  };
  load(a[0], row);
  const int32_t own = t < kSyT ? I * kSyT + t : J * kSyT + (t - kSyT);
  const double xo = ws.xtmp[min(own, n - 1)];
  double tau, scale, beta;
  col_scalars(ws, n, c, tau, scale, beta);
  if (blockIdx.x == 0 && t == 0) {
    ws.e[c] = beta;
    ws.e2[c] = beta * beta;
    ws.tau[c] = tau;
  }
  const double vo = own >= n || own <= c ? 0.0 : (own == c + 1 ? 1.0 : xo * scale);
  sv[t] = vo;
  __syncthreads();
  const double2 vc = *(const double2 *)(sv + kSyT + 2 * lane);
  double c0 = 0.0, c1 = 0.0, z[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b < 3) load(a[(b + 1) & 1], row + 8 * (b + 1));
    const double *vr = sv + 32 * wv + 8 * b;
    z[b] = diag ? symv_rows8<true>(a[b & 1], vr, row + 8 * b, col, vc.x, vc.y, c0, c1)
                : symv_rows8<false>(a[b & 1], vr, row + 8 * b, col, vc.x, vc.y, c0, c1);
  }
  {
    const bool b8 = (lane & 8) != 0, b16 = (lane & 16) != 0;
    double y = xpick(b16, xpick(b8, z[0], z[1], 8), xpick(b8, z[2], z[3], 8), 16);
    y += xlane(y, 32);
    if (lane < 32) srow[32 * wv + lane] = y;
  }
  scol[wv][2 * lane] = c0;
  scol[wv][2 * lane + 1] = c1;
  __syncthreads();
  const int i = t & (kSyT - 1);
  const double cs = (scol[0][i] + scol[1][i]) + (scol[2][i] + scol[3][i]);
  double y = t < kSyT ? srow[i] + (diag ? cs : 0.0) : (diag ? 0.0 : cs);
  if (own > c && own < n && (t < kSyT || !diag)) {
    ws.yp[(int64_t)(t < kSyT ? J : I) * lda + own] = y;
    if (diag) {
      ws.V[(int64_t)own * kNB + j] = vo;
      ws.a[(int64_t)c * lda + own] = vo;
    }
  } else {
    y = 0.0;
  }
  y = block_sum(y * vo, red);
  if (t == 0) ws.ps[blockIdx.x] = y;
}

// ---------------------------------------------------------------- wcol part
// Panel vectors are stored row-major, V[r * kNB + q], so a thread loads its row's
// coefficients in one batch; entries of columns not yet in this panel are stale
// but always meet a zero coefficient.
__device__ inline void wcol_part(const EigWs &ws, int32_t n, int32_t c, int32_t j, int32_t blk,
                                 int32_t nps) {
  __shared__ double red[4][4];
  __shared__ double pqr[4][2 * kNB];  // raw panel dots per wave
  __shared__ double pq[2 * kNB];      // p_q = V_q . v, q_q = W_q . v (zero for q >= j)
  __shared__ double cc[2 * kNB];      // V_q[c+1], W_q[c+1] (zero for q >= j)
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int sub = threadIdx.x & 3;  // this thread's quarter of the panel: q = 8 sub .. 8 sub + 7
  const int32_t c1 = c + 1;
  const int32_t lda = ws.lda;
  const double *pwc = ws.pw + (int64_t)(c & 1) * ws.maxw * kPW;
  const int32_t nw = wcol_blocks(n, c);
  // ---- all loads go out first, so the part runs on one round of memory latency: this
  // row's quarter of the panel vectors (column j is
  // rebuilt from x below) and its entry of the trailing row c+1, its x, row c+1's
  // panel coefficients, and the panel-dot and norm partials
  const int32_t r = c1 + blk * kWRows + (int32_t)(threadIdx.x >> 2);
  const bool inr = r < n;
  const int32_t rs = inr ? r : c1;  // rows past n read row c+1 (in bounds, discarded)
  // first batches of the three partial sums: panel dots (component lane over blocks
  // wv, wv+4, ..., three batches of eight), and the norm and alpha of column c
  // (blocks lane, lane+64, ...)
  double lp[3][8], ln0[8], ln1[8];
#pragma unroll
  for (int t = 0; t < 3; ++t) load8(pwc + 2 + lane, kPW, wv + 32 * t, 4, nw, lp[t]);
  load8(pwc, kPW, lane, 64, nw, ln0);
  load8(pwc + 1, kPW, lane, 64, nw, ln1);
  double vrow[8], wrow[8];
  {
    const double2 *vp = (const double2 *)(ws.V + (int64_t)rs * kNB + 8 * sub);
    const double2 *wp = (const double2 *)(ws.W + (int64_t)rs * kNB + 8 * sub);
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const double2 a2 = vp[h], b2 = wp[h];
      vrow[2 * h] = a2.x;
      vrow[2 * h + 1] = a2.y;
      wrow[2 * h] = b2.x;
      wrow[2 * h + 1] = b2.y;
    }
  }
  double base = ws.a[(int64_t)c1 * lda + rs];
  const double xr = ws.xtmp[rs];
  double atc = 0.0;
  if (threadIdx.x < 2 * kNB) {
    const int q = threadIdx.x & (kNB - 1);
    atc = (threadIdx.x < kNB) ? ws.V[(int64_t)c1 * kNB + q] : ws.W[(int64_t)c1 * kNB + q];
  }
  // the row's shares of y, four threads taking every fourth, and row c+1's, a lane each
  const int32_t nt = (n + kSyT - 1) / kSyT, i0 = c1 / kSyT;
  double ly0[8], ly1[8], yp[8];
  load8(ws.yp + rs, lda, i0 + sub, 4, nt, ly0);
  load8(ws.yp + rs, lda, i0 + sub + 32, 4, nt, ly1);
  double yc1 = ws.yp[(int64_t)min(i0 + lane, nt - 1) * lda + c1];
  yc1 = i0 + lane < nt ? yc1 : 0.0;
  for (int32_t b = i0 + lane + 64; b < nt; b += 64) yc1 += ws.yp[(int64_t)b * lda + c1];
  load8(ws.ps, 1, threadIdx.x, 256, nps, yp);
  double praw = 0.0;
  {
    const int comp = lane;  // 0..31 V dots, 32..63 W dots
    const int q = comp & (kNB - 1);
    // pairwise, so the chain is five additions long instead of 24
    double st[3];
#pragma unroll
    for (int t = 0; t < 3; ++t)
      st[t] = ((lp[t][0] + lp[t][1]) + (lp[t][2] + lp[t][3])) +
              ((lp[t][4] + lp[t][5]) + (lp[t][6] + lp[t][7]));
    praw = (st[0] + st[1]) + st[2];
    for (int32_t bb = wv + 96; bb < nw; bb += 4) praw += pwc[2 + comp + (int64_t)bb * kPW];
    praw = q < j ? praw : 0.0;
  }
  // every wave forms the scalars itself (same bits as the symv part's)
  double tau, scale;
  {
    double beta;
    col_scalars_sums(sum_rest(pwc, kPW, lane, 64, nw, ln0), sum_rest(pwc + 1, kPW, lane, 64, nw, ln1),
                     tau, scale, beta);
  }
  double yv = sum_rest(ws.ps, 1, threadIdx.x, 256, nps, yp);
  double yy = sum8(ly0) + sum_rest(ws.yp + rs, lda, i0 + sub + 32, 4, nt, ly1);
  yy += xlane(yy, 1);
  yy += xlane(yy, 2);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) yc1 += xlane(yc1, o);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) yv += xlane(yv, o);
  if (lane == 0) red[wv][0] = yv;
  pqr[wv][lane] = praw;
  __syncthreads();
  const double ydv = (red[0][0] + red[1][0]) + (red[2][0] + red[3][0]);
  if (threadIdx.x < 2 * kNB) {
    const int comp = threadIdx.x, q = comp & (kNB - 1);
    const double raw = (pqr[0][comp] + pqr[1][comp]) + (pqr[2][comp] + pqr[3][comp]);
    cc[comp] = q < j ? atc : 0.0;
    pq[comp] = q < j ? atc + scale * raw : 0.0;  // v = e_{c+1} + scale x beyond c+1
  }
  __syncthreads();
  // alpha = -tau/2 w.v with w.v = tau (y.v - 2 sum_q p_q q_q), and w_pre at row c+1
  // (same in every block).  pq and cc are zero from q = j on, so the sums run over
  // the whole panel.  Lane q (mod 32) forms term q and five exchanges (lane ^ 16 ..
  // lane ^ 1) add the terms as a tree: the same bits in every lane, wave and block.
  double spq, y1;
  {
    const int q = lane & (kNB - 1);
    double tq = pq[q] * pq[kNB + q];
    double ty = cc[q] * pq[kNB + q] + cc[kNB + q] * pq[q];
#pragma unroll
    for (int o = kNB / 2; o > 0; o >>= 1) {
      tq += xlane(tq, o);
      ty += xlane(ty, o);
    }
    spq = tq;
    y1 = yc1 - ty;
  }
  const double alpha = -0.5 * tau * (tau * (ydv - 2.0 * spq));
  const double wc1 = tau * y1;
  // the row's panel corrections: each thread sums its quarter, two exchanges add the
  // quarters (the same bits in all four threads of the row)
  {
    double py[8], pb[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int q = 8 * sub + k;
      py[k] = vrow[k] * pq[kNB + q] + wrow[k] * pq[q];
      pb[k] = cc[q] * wrow[k] + cc[kNB + q] * vrow[k];
    }
    // pairwise: three dependent additions instead of eight
    double sy = ((py[0] + py[1]) + (py[2] + py[3])) + ((py[4] + py[5]) + (py[6] + py[7]));
    double sbse = ((pb[0] + pb[1]) + (pb[2] + pb[3])) + ((pb[4] + pb[5]) + (pb[6] + pb[7]));
    sy += xlane(sy, 1);
    sbse += xlane(sbse, 1);
    sy += xlane(sy, 2);
    sbse += xlane(sbse, 2);
    yy -= sy;
    base -= sbse;
  }
  // this column's v_r, as the symv part formed it, joins vrow at j; the row's
  // W[r][j] joins wrow below
  const double vr = (r == c1) ? 1.0 : xr * scale;
#pragma unroll
  for (int k = 0; k < 8; ++k) vrow[k] = (8 * sub + k == j) ? vr : vrow[k];
  const double w = tau * yy;
  const double wj = w + alpha * vr;
  // row c+1 minus panel column j:  V[j][c1] (=1) W[j][r] + W[j][c1] V[j][r]
  const double x = base - w - wc1 * vr - 2.0 * alpha * vr;
  const bool live = inr && r >= c1 + 2;
  if (inr && sub == 0) {
    ws.W[(int64_t)r * kNB + j] = wj;
    ws.xtmp[r] = x;
    if (r == c1) ws.d[c1] = x;
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) wrow[k] = (8 * sub + k == j) ? wj : wrow[k];
  // ---- this block's partials for column c+1, summed in a fixed order:
  // norm, the next alpha (row c+2, block 0), and if column c+1 continues the
  // panel, V_q . x and W_q . x for q <= j
  const int jn = ((c1 % kNB) != 0 && c1 + 1 < n) ? j + 1 : 0;
  const double xl = live ? x : 0.0;
  double *pwn = ws.pw + (int64_t)(c1 & 1) * ws.maxw * kPW + (int64_t)blk * kPW;
  {
    double v0 = sub == 0 ? xl * xl : 0.0, v1 = (sub == 0 && inr && r == c1 + 1) ? x : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      v0 += xlane(v0, o);
      v1 += xlane(v1, o);
    }
    if (lane == 0) {
      red[wv][1] = v0;
      red[wv][2] = v1;
    }
  }
  // panel dots V_q . x, W_q . x: a thread holds 16 products (its quarter of V, then
  // of W).  Butterfly transpose-reduce over the wave's 16 rows (lane bits 5..2): the
  // exchange at offset o keeps the half selected by bit o, so lane (i, sub) ends
  // with product i (i = (lane >> 2) & 15) summed over the rows; then one pass over
  // the four waves through LDS.
  {
    double t[16];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      t[k] = vrow[k] * xl;
      t[8 + k] = wrow[k] * xl;
    }
#pragma unroll
    for (int off = 32; off >= 4; off >>= 1) {
      const int half = off >> 2;
      const bool bsel = (lane & off) != 0;
#pragma unroll
      for (int k = 0; k < half; ++k)
      {
        const double p0 = t[k], p1 = t[k + half];
        t[k] = (bsel ? p1 : p0) + xlane(bsel ? p0 : p1, off);
      }
    }
    const int i = (lane >> 2) & 15;
    const int comp = (i < 8) ? 8 * sub + i : kNB + 8 * sub + (i - 8);
    pqr[wv][comp] = t[0];
  }
  __syncthreads();
  if (threadIdx.x < 2 * kNB) {
    const int comp = threadIdx.x;
    const double sum = (pqr[0][comp] + pqr[1][comp]) + (pqr[2][comp] + pqr[3][comp]);
    pwn[2 + comp] = (comp & (kNB - 1)) < jn ? sum : 0.0;
  }
  if (threadIdx.x == 0) {
    pwn[0] = (red[0][1] + red[1][1]) + (red[2][1] + red[3][1]);
    pwn[1] = (red[0][2] + red[1][2]) + (red[2][2] + red[3][2]);
  }
}

__global__ __launch_bounds__(256) void k_wcol(EigWs ws, int32_t n, int32_t c, int32_t j, int32_t nps) {
  wcol_part(ws, n, c, j, (int32_t)blockIdx.x, nps);
}

// A[r][s] -= sum_q V[r][q] W[s][q] + W[r][q] V[s][q] for r, s >= k0: one FP64 MFMA
// GEMM with K = 2 kNB per 64x64 tile, A operand [V_r | W_r], B operand [W_s | V_s]
// (4 waves x 32x32, MFMA f64 16x16x4).
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double eig_f64x4;
constexpr int kS2K = 2 * kNB;        // GEMM depth
constexpr int kS2Ld = kS2K + 1;      // padded LDS row (conflict-free 16-row reads)

// 64 consecutive rows of two row-major n x kNB panels (P0 and P1), 16 bytes per load:
// element i of a thread covers row (t + 256 i) / 16, columns 2 ((t + 256 i) % 16) + {0, 1}.
// Rows at or past n load row n - 1 and are zeroed when stored.
struct S2Rows {
  double2 p[2][4];
};
__device__ __forceinline__ void s2_load(const double *P0, const double *P1, int32_t r0,
                                        int32_t n, S2Rows &s) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = threadIdx.x + 256 * i;
    const int64_t off = (int64_t)min(r0 + (e >> 4), n - 1) * kNB + 2 * (e & 15);
    s.p[0][i] = *(const double2 *)(P0 + off);
    s.p[1][i] = *(const double2 *)(P1 + off);
  }
}
// row o of `sm`: P0's kNB columns, then P1's; columns at or past nb are zero
__device__ __forceinline__ void s2_store(double (*sm)[kS2Ld], int32_t r0, int32_t n,
                                         int32_t nb, const S2Rows &s) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = threadIdx.x + 256 * i, o = e >> 4, q = 2 * (e & 15);
    const bool ok = r0 + o < n;
    const bool ok0 = ok && q < nb, ok1 = ok && q + 1 < nb;
    sm[o][q] = ok0 ? s.p[0][i].x : 0.0;
    sm[o][q + 1] = ok1 ? s.p[0][i].y : 0.0;
    sm[o][kNB + q] = ok0 ? s.p[1][i].x : 0.0;
    sm[o][kNB + q + 1] = ok1 ? s.p[1][i].y : 0.0;
  }
}

// One block per 64x64 tile of the upper triangle (all that is read).  The B operand rows [W_c | V_c] are staged in LDS; each
// lane's A operand stays in registers: the MFMA sums over k, so lane group g = lane / 16
// takes k = 16 g + ks at step ks (in A and B alike), and its A entries are 16
// consecutive doubles of a row of V (g < 2) or W.  33 KB of LDS and ~150 registers
// give three blocks per CU.
__global__ __launch_bounds__(256) void k_syr2k(EigWs ws, int32_t n, int32_t k0, int32_t nb) {
  __shared__ double sb[64][kS2Ld];
  const int32_t nt = (n - k0 + 63) / 64;
  int32_t tr, tc;
  upper_tile((int32_t)blockIdx.x, nt, tr, tc);
  const int32_t rb = k0 + tr * 64, cb = k0 + tc * 64;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wr = w >> 1, wc = w & 1, g = lane >> 4;
  const int32_t lda = ws.lda;
  // the B rows and the A entries are loaded together (both from L2-resident panels)
  S2Rows rbv;
  s2_load(ws.W, ws.V, cb, n, rbv);
  double2 av2[2][8];
  {
    const double *asrc = (g < 2 ? ws.V : ws.W) + 16 * (g & 1);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      // rows past n read row n - 1 (their results are not stored)
      const int32_t r = min(rb + 32 * wr + 16 * a + (lane & 15), n - 1);
      const double2 *src = (const double2 *)(asrc + (int64_t)r * kNB);
#pragma unroll
      for (int h = 0; h < 8; ++h) av2[a][h] = src[h];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load goes out before the LDS stores wait
  s2_store(sb, cb, n, nb, rbv);
  // panel columns at or past nb take no part (zero in A as in B)
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const int q = 16 * (g & 1) + 2 * h;
      av2[a][h].x = q < nb ? av2[a][h].x : 0.0;
      av2[a][h].y = q + 1 < nb ? av2[a][h].y : 0.0;
    }
  __syncthreads();
  // the tile's old values (row, column of lane's accumulator elements) load while the
  // products are formed; indices past n are clamped, and those elements are never stored
  double old[2][2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int32_t r = min(rb + 32 * wr + 16 * a + (lane >> 4) + 4 * e, n - 1);
        const int32_t c = min(cb + 32 * wc + 16 * b + (lane & 15), n - 1);
        old[a][b][e] = ws.a[(int64_t)r * lda + c];
      }
  __builtin_amdgcn_sched_barrier(0);  // the old values are in flight before the first product
  eig_f64x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = eig_f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int ks = 0; ks < 16; ++ks) {
    double bv[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) bv[b] = sb[32 * wc + 16 * b + (lane & 15)][16 * g + ks];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const double av = (ks & 1) ? av2[a][ks >> 1].y : av2[a][ks >> 1].x;
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[b], acc[a][b], 0, 0, 0);
    }
  }
  // accumulator layout: lane l, element e -> row l/16 + 4e, column l%16
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int32_t r = rb + 32 * wr + 16 * a + (lane >> 4) + 4 * e;
        const int32_t c = cb + 32 * wc + 16 * b + (lane & 15);
        if (r < n && c < n) ws.a[(int64_t)r * lda + c] = old[a][b][e] - acc[a][b][e];
      }
}

// ---------------------------------------------------------------- resident part
// Tridiagonalisation of a trailing matrix that the register files hold: columns c0 .. c1-1
// in one launch, block b holding rows c0 + b RS .. in registers (thread t: columns c0 + t +
// T k of every row).  Per column c every block forms the same reflector v from x = row c
// and the products of its own rows with it; they and the owner's copy of row c+1 go to
// memory, every block reads all of them back and forms w = tau y + alpha v and the next x
// = row c+1 - w - w_{c+1} v for itself, and each applies the rank-2 update to its own rows
// while it forms the next products.  So a column is one exchange between blocks, three
// barriers within them, and no pass over memory.
//
// Every word exchanged is its own flag: the buffers hold kTriNone, a NaN that no
// arithmetic produces, until the word's one store of the launch (device-coherent, 8 bytes
// at once), and a reader polls the words it needs with device-coherent loads until none is
// kTriNone.  No order between words is assumed.  A block whose rows are all done leaves.
// The blocks have to run at the same time: there is one per CU at most (host side), and
// the host runs one such launch at a time on a device (two that each held part of the CUs
// would wait for each other).  Should some not be scheduled (the
// device shared with other programs), each wait ends after kTriLimit ticks of the wall
// clock and sets sync[1]; the host then starts over without this kernel.
constexpr uint64_t kTriNone = 0xFFF4E1D2C3B4A596ull;
constexpr int64_t kTriLimit = 50000000;  // 0.5 s at 100 MHz
__global__ __launch_bounds__(256) void k_tri_fill(uint64_t *__restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    p[i] = kTriNone;
}
__device__ __forceinline__ void store_dev(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double load_dev(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Sums over the wave of the row values that lanes hold, four rows at a time as they come
// (few registers live at once), then over the groups: lane l ends with row l % R2's sum
// (R2 = 8 or 16).  rows4 leaves row l % 4 summed over the lanes' groups of four.
__device__ __forceinline__ double rows4(const double (&v)[4]) {
  const int lane = threadIdx.x & 63;
  const bool b2 = (lane & 2) != 0, b1 = (lane & 1) != 0;
  return xpick(b1, xpick(b2, v[0], v[2], 2), xpick(b2, v[1], v[3], 2), 1);
}
template <int G>
__device__ __forceinline__ double rows_sum(const double (&z)[G]) {
  const int lane = threadIdx.x & 63;
  const bool b4 = (lane & 4) != 0, b8 = (lane & 8) != 0;
  double a;
  if constexpr (G == 1) {
    a = z[0];
    a += xlane(a, 4);
    a += xlane(a, 8);
  } else if constexpr (G == 2) {
    a = xpick(b4, z[0], z[1], 4);
    a += xlane(a, 8);
  } else {
    const double z3 = G == 4 ? z[G - 1] : 0.0;
    a = xpick(b4, xpick(b8, z[0], z[2], 8), xpick(b8, z[1], z3, 8), 4);
  }
  a += xlane(a, 16);
  a += xlane(a, 32);
  return a;
}
// 1/a by the hardware reciprocal and two Newton steps (error a few ulp)
__device__ __forceinline__ double rcp_nr(double a) {
  double r = __builtin_amdgcn_rcp(a);
  r = fma(r, fma(-a, r, 1.0), r);
  return fma(r, fma(-a, r, 1.0), r);
}
// Indices are local to the stage: column and row i of the kernel are c0 + i of the matrix.
template <int T, int K, int RS>
__global__ __launch_bounds__(T) void k_tri(EigWs ws, int32_t n, int32_t c0, int32_t c1,
                                           double *__restrict__ yb, double *__restrict__ rb,
                                           int64_t ldb) {
  constexpr int W = T / 64;
  constexpr int G = RS / 4;  // rows are summed in groups of four
  static_assert(RS % 4 == 0 && RS <= 16, "rows per block");
  __shared__ double sv[2][T * K], sw[T * K];
  __shared__ double red[W][16], rdot[W], rnrm[W], sy1, sal;
  __shared__ int32_t dead;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int32_t nl = n - c0, cols = c1 - c0, r0 = (int32_t)blockIdx.x * RS;  // first row
  const int64_t lda = ws.lda;
  double *const A = ws.a + (int64_t)c0 * lda + c0;
  // thread t's columns are t + T k: with the uniform part in scalars, one offset serves all
  // of a thread's addresses, and comparisons are with t
  double a[RS][K], x[K], v[K], w[K];
#pragma unroll
  for (int s = 0; s < RS; ++s)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int32_t r = min(r0 + s, nl - 1), q = min(t + T * k, nl - 1);  // upper triangle
      const double z = A[(int64_t)min(r, q) * lda + max(r, q)];
      a[s][k] = (r0 + s < nl && t < nl - T * k) ? z : 0.0;
    }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double *p = A + T * k;
    x[k] = t < nl - T * k ? p[t] : 0.0;
    v[k] = w[k] = 0.0;
    sv[0][t + T * k] = sv[1][t + T * k] = sw[t + T * k] = 0.0;
  }
  if (t == 0) dead = 0;
  if (blockIdx.x == 0 && t == 0) ws.d[c0] = x[0];
  // row c is overwritten by its reflector only after an exchange that every block took part
  // in, so each has read row c0 and its own rows by then
  // norm of x beyond c + 1, and x_{c+1}
  auto norm = [&](int32_t c) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      s = fma(x[k], t >= c + 2 - T * k ? x[k] : 0.0, s);
      if (t == c + 1 - T * k) sal = x[k];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += xlane(s, o);
    if (lane == 0) rnrm[wv] = s;
  };
  norm(0);
  // 2^-160 of the largest squared norm of a column, first of those before this launch
  {
    double top = 0.0;
    for (int32_t i = t; i < c0; i += T) top = fmax(top, 0x1p-160 * ws.e2[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmax(top, xlane(top, o));
    if (lane == 0) rdot[wv] = top;
  }
  __syncthreads();
  double drop = rdot[0];
#pragma unroll
  for (int u = 1; u < W; ++u) drop = fmax(drop, rdot[u]);
  for (int32_t c = 0; c < cols; ++c) {
    if (r0 + RS - 1 <= c) return;  // no live rows: nothing to give and nothing to keep
    const int cur = c & 1;
    // ---- the reflector of column c (dlarfg), the same in every block
    double xn2 = rnrm[0];
#pragma unroll
    for (int u = 1; u < W; ++u) xn2 += rnrm[u];
    const double al = sal;
    double tau = 0.0, scale = 0.0, beta = al;
    // A matrix of constant blocks leaves a remainder of the same structure in every column,
    // each 1e-16 of the last, until its squares underflow and tau no longer fits v (vectors
    // orthogonal to 1e-2 only).  What is below 2^-80 of an earlier column is far below the
    // matrix' rounding: it is dropped, as the Sturm counts do with such an e.
    if (xn2 > drop) {
      const double s2 = fma(al, al, xn2);
      if (s2 > 1e-280 && s2 < 1e280) {
        // 1 / sqrt and 1 / x by the hardware's approximations and two Newton steps each (a
        // few ulps, as rcp_nr's), whose chains are shorter than a square root's and division's
        double h = __builtin_amdgcn_rsq(s2);
        h = fma(h, fma(-0.5 * s2 * h, h, 0.5), h);
        h = fma(h, fma(-0.5 * s2 * h, h, 0.5), h);
        const double nb = copysign(s2 * h, al);  // -beta
        beta = -nb;
        tau = fma(fabs(al), h, 1.0);
        scale = rcp_nr(al + nb);
      } else {
        beta = -copysign(sqrt(s2), al);
        tau = (beta - al) / beta;
        scale = 1.0 / (al - beta);
      }
    }
    double vn[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int32_t p = c + 1 - T * k;
      vn[k] = t == p ? 1.0 : (t > p ? x[k] * scale : 0.0);
      sv[cur][t + T * k] = vn[k];
    }
    // ---- the update by column c - 1 (v, w; zero at first) and the products with vn
    double z[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = 4 * g + u;
        const double vi = sv[cur ^ 1][r0 + s], wi = sw[r0 + s];
#pragma unroll
        for (int k = 0; k < K; ++k) {
          a[s][k] = fma(-vi, w[k], fma(-wi, v[k], a[s][k]));
          acc[u] = fma(a[s][k], vn[k], acc[u]);
        }
      }
      z[g] = rows4(acc);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- row c + 1 to the others
    const bool owner = c + 1 >= r0 && c + 1 < r0 + RS;
    double *const rrow = rb + (int64_t)c * ldb, *const yrow = yb + (int64_t)c * ldb;
    if (owner) {
#pragma unroll
      for (int s = 0; s < RS; ++s)
        if (c + 1 == r0 + s)
#pragma unroll
          for (int k = 0; k < K; ++k)
            if (t > c - T * k && t < nl - T * k) store_dev(rrow + T * k + t, a[s][k]);
    }
    {
      const double rs = rows_sum<G>(z);
      if (lane < 16) red[wv][lane] = rs;
    }
    __syncthreads();
    if (t < RS && r0 + t > c && r0 + t < nl) {
      double y = red[0][t];
#pragma unroll
      for (int u = 1; u < W; ++u) y += red[u][t];
      store_dev(yrow + r0 + t, y);
    }
    // ---- everyone's products and row c + 1
    {
      double *const y = w, *const r = x;  // their registers
      int64_t t_end = 0;
      for (int32_t spin = 0;; ++spin) {
        bool all = true;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          y[k] = r[k] = 0.0;
          if (t > c - T * k && t < nl - T * k) {
            y[k] = load_dev(yrow + T * k + t);
            r[k] = load_dev(rrow + T * k + t);
          }
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
          all = all && __builtin_bit_cast(uint64_t, y[k]) != kTriNone &&
                __builtin_bit_cast(uint64_t, r[k]) != kTriNone;
        if (all) break;
        if ((spin & 255) == 255) {
          const int64_t now = (int64_t)wall_clock64();
          if (t_end == 0) t_end = now + kTriLimit;
          if (now > t_end ||
              __hip_atomic_load(ws.sync + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
            dead = 1;
            break;
          }
        }
      }
    }
    double dt = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      dt = fma(w[k], vn[k], dt);
      if (t == c + 1 - T * k) sy1 = w[k];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dt += xlane(dt, o);
    if (lane == 0) rdot[wv] = dt;
    __syncthreads();
    if (dead) {
      if (t == 0) __hip_atomic_store(ws.sync + 1, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    double ydv = rdot[0];
#pragma unroll
    for (int u = 1; u < W; ++u) ydv += rdot[u];
    // w = tau y + alpha v (y and v are zero up to column c), x = row c + 1 - w - w_{c+1} v
    const double alpha = -0.5 * tau * (tau * ydv);
    const double w1 = tau * sy1 + alpha;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      v[k] = vn[k];
      w[k] = tau * w[k] + alpha * vn[k];
      x[k] = x[k] - w[k] - w1 * vn[k];
      sw[t + T * k] = w[k];
    }
    norm(c + 1);
    drop = fmax(drop, 0x1p-160 * (beta * beta));
    // ---- results of column c, by the owner of row c + 1
    if (owner) {
      double *const out = A + (int64_t)c * lda;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (t > c - T * k && t < nl - T * k) (out + T * k)[t] = vn[k];
        if (t == c + 1 - T * k) ws.d[c0 + c + 1] = x[k];
      }
      if (t == 0) {
        ws.e[c0 + c] = beta;
        ws.e2[c0 + c] = beta * beta;
        ws.tau[c0 + c] = tau;
      }
    }
    __syncthreads();
  }
  // the last update, and the rows back to memory for what follows
  if (c1 >= n - 1) return;
  const int last = (cols - 1) & 1;
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const double vi = sv[last][r0 + s], wi = sw[r0 + s];
    if (r0 + s < cols || r0 + s >= nl) continue;
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (t >= cols - T * k && t < nl - T * k)
        (A + (int64_t)(r0 + s) * lda + T * k)[t] = fma(-vi, w[k], fma(-wi, v[k], a[s][k]));
  }
}

// ---------------------------------------------------------------- eigenvalues
__global__ void k_gersh(EigWs ws, int32_t n) {
  __shared__ double lo[256], hi[256], mx[256], tnr[256];
  double gl = 1e300, gu = -1e300, emax = 0.0, tn = 0.0;
  for (int32_t i = threadIdx.x; i < n; i += blockDim.x) {
    double r = 0.0;
    if (i > 0) r += fabs(ws.e[i - 1]);
    if (i < n - 1) r += fabs(ws.e[i]);
    gl = fmin(gl, ws.d[i] - r);
    gu = fmax(gu, ws.d[i] + r);
    if (i < n - 1) emax = fmax(emax, ws.e2[i]);
    tn = fmax(tn, fabs(ws.d[i]) + r);
  }
  lo[threadIdx.x] = gl;
  hi[threadIdx.x] = gu;
  mx[threadIdx.x] = emax;
  tnr[threadIdx.x] = tn;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      lo[threadIdx.x] = fmin(lo[threadIdx.x], lo[threadIdx.x + o]);
      hi[threadIdx.x] = fmax(hi[threadIdx.x], hi[threadIdx.x + o]);
      mx[threadIdx.x] = fmax(mx[threadIdx.x], mx[threadIdx.x + o]);
      tnr[threadIdx.x] = fmax(tnr[threadIdx.x], tnr[threadIdx.x + o]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double eps = 2.220446049250313e-16, safmin = 2.2250738585072014e-308;
    double tnorm = fmax(fabs(lo[0]), fabs(hi[0]));
    double pivmin = safmin * fmax(1.0, mx[0]);
    ws.sc[S_GL] = lo[0] - 2.0 * eps * tnorm * n - 2.0 * pivmin;
    ws.sc[S_GU] = hi[0] + 2.0 * eps * tnorm * n + 2.0 * pivmin;
    ws.sc[S_PIVMIN] = pivmin;
    ws.sc[S_TNORM] = fmax(tnr[0], 1e-300);
    ws.sc[S_SCALE] = ldexp(1.0, -ilogb(ws.sc[S_TNORM]) - 1);
  }
}

// T over a power of two of its norm, as the Sturm counts read it: (d_i, e_{i-1}^2) in steps
// of 2 kStB, the last ones filled with rows that change no sign, and one batch more that is
// read ahead.  e^2 is kept at 2^-160 at least (2^-80 of the norm, far below an eigenvalue's
// rounding), so that a zero minor is followed by one that is not.
constexpr int kStB = 8;
__host__ __device__ inline int32_t sturm_rows(int32_t n) { return (n + 2 * kStB - 1) / (2 * kStB) * (2 * kStB); }
__global__ __launch_bounds__(256) void k_sturm_prep(EigWs ws, int32_t n) {
  const int32_t i = (int32_t)(blockIdx.x * 256 + threadIdx.x);
  if (i >= sturm_rows(n) + kStB) return;
  const double s = ws.sc[S_SCALE];
  double2 v = make_double2(8.0, 0x1p-160);
  if (i < n) {
    v.x = ws.d[i] * s;
    const double e = i > 0 ? ws.e[i - 1] * s : 0.0;
    v.y = fmax(e * e, 0x1p-160);
  }
  ws.st[i] = v;
}

// the block pulls T into its L2 together: scalar loads that miss there one batch after the
// other took 47 ns a step of a launch's first count
__device__ __forceinline__ void sturm_warm(const double2 *__restrict__ T, int32_t n) {
  for (int32_t i = kStB * (int32_t)threadIdx.x; i < n; i += kStB * 256) {
    const double v = T[i].x;
    asm volatile("" ::"v"(v));
  }
}

// Number of eigenvalues of T below x: the sign changes in the sequence of leading minors
// p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2} of the scaled T - x I.  Only its one fused
// multiply-add is on the chain from step to step (the recurrence of quotients has a
// reciprocal there: 78 cycles a step, now 35); each step's rounding amounts to a relative
// change of d_i - x and of e_{i-1}^2.  A batch grows by at most 2^16 and shrinks by 2^-640 or
// so where minors vanish, and is followed by a common scaling of the last two.  Signs are
// shifted into a word and their changes counted per batch.  d and e^2 are wave-uniform
// (scalar) loads, one batch ahead of use.
__device__ inline int32_t sturm1(const double2 *T2, int32_t n, double x) {
  // constant address space: uniform reads of it are scalar loads
  typedef const __attribute__((address_space(4))) double *Scalars;
  const Scalars T = (Scalars)(uintptr_t)T2;
  int32_t cnt = 0;
  uint32_t bits = 0;
  double p1 = 1.0, p2 = 0.0;
  auto run = [&](const double (&v)[2 * kStB]) {
#pragma unroll
    for (int u = 0; u < kStB; ++u) {
      const double p = fma(v[2 * u] - x, p1, -(v[2 * u + 1] * p2));
      p2 = p1;
      p1 = p;
      bits = __builtin_amdgcn_alignbit(bits, (uint32_t)__double2hiint(p), 31);
    }
    cnt += __popc((bits ^ (bits >> 1)) & ((1u << kStB) - 1u));
    const double m = fmax(fabs(p1), fabs(p2));
    const int ex = __builtin_amdgcn_frexp_exp(m);
    p1 = m > 0.0 ? __builtin_amdgcn_ldexp(p1, -ex) : 1.0;
    p2 = __builtin_amdgcn_ldexp(p2, -ex);
  };
  // the loads of v, once those of w have arrived (scalar loads end in any order, so a wait is
  // for all that are out)
  auto ld = [&](int32_t i, double (&v)[2 * kStB], const double (&w)[2 * kStB]) {
    asm volatile("" ::"s"(w[0]), "s"(w[2 * kStB - 1]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2 * kStB; ++u) v[u] = T[2 * i + u];
    __builtin_amdgcn_sched_barrier(0);  // not moved down to their use
  };
  double a[2 * kStB], b[2 * kStB];
#pragma unroll
  for (int u = 0; u < 2 * kStB; ++u) a[u] = T[u];
  const int32_t rows = sturm_rows(n);
  for (int32_t i = 0; i < rows; i += 2 * kStB) {
    ld(i + kStB, b, a);
    run(a);
    ld(i + 2 * kStB, a, b);
    run(b);
  }
  return cnt;
}

// Shared first level: Sturm counts at kMsGrid evenly spaced interior points of the
// Gershgorin interval, one per thread (each a count over the whole tridiagonal, like
// one round of the multisection for kMsGrid / 16 eigenvalues).  Every eigenvalue then
// starts from the grid interval that brackets it, kMsGrid + 1 times narrower than the
// Gershgorin interval, which saves about four rounds.
constexpr int kMsGrid = 65536;
__device__ __forceinline__ double msgrid_x(double glo, double ghi, int32_t j) {
  return glo + (ghi - glo) / (double)(kMsGrid + 1) * (double)(j + 1);
}
__global__ __launch_bounds__(256) void k_msgrid(EigWs ws, int32_t n, int32_t *__restrict__ gcnt) {
  const int32_t j = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);  // kMsGrid threads
  sturm_warm(ws.st, n);
  gcnt[j] = sturm1(ws.st, n, msgrid_x(ws.sc[S_GL], ws.sc[S_GU], j) * ws.sc[S_SCALE]);
}
// kMS lanes per eigenvalue (k-th smallest): each round the lanes evaluate kMS interior
// points of [lo, hi] and keep the sub-interval holding eigenvalue k.  One count per lane.  A
// round takes the same time while the waves fit one per SIMD and more lanes save rounds, so
// the launch takes 64 lanes up to order 1,024 and halves them for every doubling, down to 8;
// with more waves than SIMDs a round's work counts.  With the counts' grid: order 198 108 ->
// 33 us, 1,000 490 -> 125, 1,203 590 -> 180, 5,000 2.46 -> 1.05 ms.
// gcnt: k_msgrid's counts, or null to start from the Gershgorin interval
template <int kMS>
__global__ __launch_bounds__(256) void k_multisect(EigWs ws, int32_t n,
                                                   const int32_t *__restrict__ gcnt) {
  const int32_t k = (int32_t)((blockIdx.x * blockDim.x + threadIdx.x) / kMS);
  const int sub = threadIdx.x % kMS;
  const bool active = k < n;
  double lo = ws.sc[S_GL], hi = ws.sc[S_GU];
  if (gcnt != nullptr && active) {
    // the grid interval bracketing eigenvalue k: a ends as a point (or the lower bound,
    // a = -1) whose count is <= k, b as one (or the upper bound, b = kMsGrid) whose
    // count is > k, adjacent -- a valid start whatever the counts' rounding
    int32_t a = -1, b = kMsGrid;
    while (b - a > 1) {
      const int32_t m = (a + b) >> 1;
      if (gcnt[m] <= k) a = m; else b = m;
    }
    const double glo = lo, ghi = hi;
    if (a >= 0) lo = msgrid_x(glo, ghi, a);
    if (b < kMsGrid) hi = msgrid_x(glo, ghi, b);
  }
  const double pivmin = ws.sc[S_PIVMIN];
  const double eps = 2.220446049250313e-16;
  // absolute floor eps * ||T||_1, the default of LAPACK's dstebz (ABSTOL <= 0): an
  // eigenvalue at zero (the centred matrix has one) converges in ~13 rounds instead
  // of running to the round cap with a relative tolerance alone
  const double atol = eps * ws.sc[S_TNORM];
  sturm_warm(ws.st, n);
  for (int it = 0; it < 96; ++it) {
    const double tol = 2.0 * eps * fmax(fabs(lo), fabs(hi)) + 4.0 * pivmin + atol;
    const bool done = (hi - lo <= tol);
    // all kMS lanes of a group share lo/hi, so `done` is uniform within a group
    if (__all(done || !active)) break;
    const double w = (hi - lo) / (double)(kMS + 1);
    const double x = lo + w * (double)(sub + 1);
    int32_t cnt = 0;
    if (active && !done) cnt = sturm1(ws.st, n, x * ws.sc[S_SCALE]);
    // new lo = largest point with count <= k ; new hi = smallest point with count > k
    double cand_lo = (cnt <= k) ? x : -1e300;
    double cand_hi = (cnt > k) ? x : 1e300;
    for (int o = kMS / 2; o > 0; o >>= 1) {
      cand_lo = fmax(cand_lo, __shfl_xor(cand_lo, o, kMS));
      cand_hi = fmin(cand_hi, __shfl_xor(cand_hi, o, kMS));
    }
    if (!done) {
      double nlo = fmax(lo, cand_lo), nhi = fmin(hi, cand_hi);
      if (nhi < nlo) nhi = nlo;
      lo = nlo;
      hi = nhi;
    }
  }
  if (active && sub == 0) ws.eval[k] = 0.5 * (lo + hi);
}

// ---------------------------------------------------------------- inverse iteration
// The LU of T - lambda I keeps pivot reciprocals, so no division sits on a serial chain.

// The shift for eigenvalue i (ascending) of the n: the eigenvalue itself, unless it belongs to a
// run of ones that stand closer than their own errors (8 ulps of the norm apart).  Shifts that
// differ by such an error turn the run's vectors to whichever of its directions is nearest to
// each, several to the same one, and orthogonalising them again leaves rounding errors
// enlarged a hundred times and more: residuals of 1e-13 where an eigenvalue fills several batches of
// vectors.  The whole run (at most 32 ulps wide) takes one shift instead, 16 of its widths off
// its middle: a solve scales all of its directions alike, so vectors orthogonalised after the
// first one stay so in the second.  Other directions shrink by 16 widths over the gap to the
// next eigenvalue a solve; where that is above 1e-10 the eigenvalues keep their own shifts.
// Every lane of a wave calls it with the same i.
__device__ inline double invit_shift(const double *__restrict__ eval, int32_t n, int32_t i, double tnorm) {
  const double ulp = 2.220446049250313e-16 * tnorm, lam = eval[i];
  auto apart = [&](int32_t k) { return k < 0 || k + 1 >= n || !(eval[k + 1] - eval[k] <= 8.0 * ulp); };
  if (apart(i - 1) && apart(i)) return lam;
  const int lane = threadIdx.x & 63;
  int32_t a = i, b = i;  // the run's ends, 64 steps at a time
  for (;; a -= 64) {
    const uint64_t m = __ballot(apart(a - 1 - lane));
    if (m == 0) continue;
    a -= __ffsll((unsigned long long)m) - 1;
    break;
  }
  for (;; b += 64) {
    const uint64_t m = __ballot(apart(b + lane));
    if (m == 0) continue;
    b += __ffsll((unsigned long long)m) - 1;
    break;
  }
  const double width = fmax(eval[b] - eval[a], 2.0 * ulp);
  double gap = tnorm;
  if (a > 0) gap = fmin(gap, eval[a] - eval[a - 1]);
  if (b + 1 < n) gap = fmin(gap, eval[b + 1] - eval[b]);
  const double off = 16.0 * width;
  return width <= 32.0 * ulp && off <= 1e-10 * gap ? 0.5 * (eval[a] + eval[b]) + off : lam;
}

// One inverse iteration for the eigenvalues j0 + blockIdx.x (descending order) of the
// tridiagonal, one block per vector: with `first` from a fixed start vector, else from
// X[j]; the pivoted LU of T - lambda I is formed with `factor`, else read back; the result is
// normalised.  The three recurrences (LU, forward, backward) are serial, about 130, 40 and 40
// cycles a step by their chains, and the rest has to stay off them: kInvC steps at a time are
// brought to LDS by the whole block, one lane runs them there, kInvB steps of operands read
// ahead, and the block writes the results back in whole lines.  The forward solve of a
// factoring pass runs in the LU's loop, behind its longer chain.  A lane per vector with its
// loads and stores in global memory, sixteen steps ahead, spent 0.65 us a row on two
// iterations of ten vectors (every store had to end before a later load counted).
//
// The LU factors: field f of step i of block b at lu[(b kLuF + f) n + i] (f: 0 pivot
// reciprocal, 1 and 2 the U superdiagonals, 3 multiplier, 4 pivot flag).
constexpr int kLuF = 5;
constexpr int kInvB = 8;
constexpr int kInvC = 512;
__global__ __launch_bounds__(256) void k_invit_solve(EigWs ws, int32_t n, int32_t j0, int32_t first,
                                                     int32_t factor, double *__restrict__ X,
                                                     double *__restrict__ lu) {
  // fields 0-4 as above (d and e come in as 0 and 1), 5 x; entry kInvC of field 1 is the e
  // after the chunk
  __shared__ __align__(16) double f[kLuF + 1][kInvC + 2];
  __shared__ double red[4], sinv;
  const int tid = threadIdx.x;
  const int32_t j = j0 + (int32_t)blockIdx.x;
  const double lam = factor ? invit_shift(ws.eval, n, n - 1 - j, ws.sc[S_TNORM]) : 0.0;
  const double tiny = 2.220446049250313e-16 * ws.sc[S_TNORM];
  double *x = X + (int64_t)j * n, *L = lu + (int64_t)blockIdx.x * kLuF * n;
  // start vectors: a fixed hash of index and vector
  auto start = [&](int32_t i) {
    uint32_t h = (uint32_t)(i + 1) * 2654435761u ^ (uint32_t)(j + 7) * 40503u;
    h ^= h >> 15; h *= 2246822519u; h ^= h >> 13;
    return 0.5 + (double)(h & 0xFFFFFF) / 16777216.0;
  };
  // ---- LU and forward solve P L: step i works on rows i and i + 1.  Lane 0 carries the
  // current row (acur, bcur) and x from chunk to chunk
  double acur = ws.d[0] - lam, bcur = n > 1 ? ws.e[0] : 0.0;
  double carry = first ? start(0) : x[0];
  for (int32_t c0 = 0; c0 < n - 1; c0 += kInvC) {
    const int32_t m = min(kInvC, n - 1 - c0);  // steps of this chunk
    for (int32_t i = tid; i < kInvC; i += 256) {
      const bool in = i < m;
      const int32_t g = in ? c0 + i : n - 2;
      if (factor) {
        f[0][i] = ws.d[g + 1];
        f[1][i] = ws.e[g];
      } else {
        f[3][i] = L[3 * (int64_t)n + g];
        f[4][i] = L[4 * (int64_t)n + g];
      }
      f[5][i] = first ? start(g + 1) : x[g + 1];
    }
    if (tid == 0) f[1][kInvC] = c0 + kInvC < n - 1 ? ws.e[c0 + kInvC] : 0.0;
    __syncthreads();
    if (tid == 0) {
      if (factor) {
        // the e after the last step is outside the recurrence
        if (m < kInvC) f[1][m] = 0.0;
        double db[kInvB], eb[kInvB], xb[kInvB], dn[kInvB], en[kInvB], xn[kInvB];
        auto ld = [&](int32_t i, double (&d)[kInvB], double (&e)[kInvB], double (&y)[kInvB]) {
          i = min(i, kInvC - kInvB);
#pragma unroll
          for (int k = 0; k < kInvB; ++k) {
            d[k] = f[0][i + k];
            e[k] = f[1][i + k + 1];
            y[k] = f[5][i + k];
          }
        };
        double l = f[1][0];
        auto run = [&](bool full, int32_t i0, const double (&d)[kInvB], const double (&e)[kInvB],
                       const double (&y)[kInvB]) {
#pragma unroll
          for (int k = 0; k < kInvB; ++k) {
            const int32_t i = i0 + k;
            if (full || i < m) {
              const double an = d[k] - lam, bn = e[k];
              const bool sw = fabs(acur) < fabs(l);  // row interchange
              const double a0 = fabs(acur) < tiny ? copysign(tiny, acur == 0.0 ? 1.0 : acur) : acur;
              const double r = rcp_nr(sw ? l : a0);
              const double mu = (sw ? acur : l) * r;
              f[0][i] = r;
              f[1][i] = sw ? an : bcur;
              f[2][i] = sw ? bn : 0.0;
              f[3][i] = mu;
              f[4][i] = sw ? 1.0 : 0.0;
              const double na = sw ? bcur - mu * an : an - mu * bcur;
              bcur = sw ? -mu * bn : bn;
              acur = na;
              l = bn;
              const double lo = sw ? y[k] : carry, nx = sw ? carry : y[k];
              f[5][i] = lo;
              carry = nx - mu * lo;
            }
          }
        };
        // a batch is read before the one ahead of it is written: no step reads what an
        // earlier one wrote
        ld(0, db, eb, xb);
        for (int32_t i0 = 0; i0 < m; i0 += 2 * kInvB) {
          ld(i0 + kInvB, dn, en, xn);
          if (i0 + kInvB <= m) run(true, i0, db, eb, xb); else run(false, i0, db, eb, xb);
          ld(i0 + 2 * kInvB, db, eb, xb);
          if (i0 + 2 * kInvB <= m) run(true, i0 + kInvB, dn, en, xn); else run(false, i0 + kInvB, dn, en, xn);
        }
      } else {
        double mb[kInvB], pb[kInvB], xb[kInvB], mn[kInvB], pn[kInvB], xn[kInvB];
        auto ld = [&](int32_t i, double (&u)[kInvB], double (&p)[kInvB], double (&y)[kInvB]) {
          i = min(i, kInvC - kInvB);
#pragma unroll
          for (int k = 0; k < kInvB; ++k) {
            u[k] = f[3][i + k];
            p[k] = f[4][i + k];
            y[k] = f[5][i + k];
          }
        };
        auto run = [&](bool full, int32_t i0, const double (&u)[kInvB], const double (&p)[kInvB],
                       const double (&y)[kInvB]) {
#pragma unroll
          for (int k = 0; k < kInvB; ++k) {
            const int32_t i = i0 + k;
            if (full || i < m) {
              const bool sw = p[k] != 0.0;
              const double lo = sw ? y[k] : carry, nx = sw ? carry : y[k];
              f[5][i] = lo;
              carry = nx - u[k] * lo;
            }
          }
        };
        ld(0, mb, pb, xb);
        for (int32_t i0 = 0; i0 < m; i0 += 2 * kInvB) {
          ld(i0 + kInvB, mn, pn, xn);
          if (i0 + kInvB <= m) run(true, i0, mb, pb, xb); else run(false, i0, mb, pb, xb);
          ld(i0 + 2 * kInvB, mb, pb, xb);
          if (i0 + 2 * kInvB <= m) run(true, i0 + kInvB, mn, pn, xn); else run(false, i0 + kInvB, mn, pn, xn);
        }
      }
    }
    __syncthreads();
    for (int32_t i = tid; i < m; i += 256) {
      if (factor)
#pragma unroll
        for (int k = 0; k < kLuF; ++k) L[k * (int64_t)n + c0 + i] = f[k][i];
      x[c0 + i] = f[5][i];
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (factor) {
      if (fabs(acur) < tiny) acur = copysign(tiny, acur == 0.0 ? 1.0 : acur);
      L[n - 1] = rcp_nr(acur);
      L[2 * (int64_t)n - 1] = L[3 * (int64_t)n - 1] = 0.0;
    }
    x[n - 1] = carry;
  }
  __syncthreads();
  // ---- backward solve U, chunks from the end
  double x1 = 0.0, x2 = 0.0, ss = 0.0;
  for (int32_t e0 = n; e0 > 0; e0 -= kInvC) {
    const int32_t c0 = max(0, e0 - kInvC), m = e0 - c0;
    for (int32_t i = tid; i < m; i += 256) {
#pragma unroll
      for (int k = 0; k < 3; ++k) f[k][i] = L[k * (int64_t)n + c0 + i];
      f[5][i] = x[c0 + i];
    }
    __syncthreads();
    if (tid == 0) {
      double yb[kInvB], ab[kInvB], bb[kInvB], cb[kInvB], yn[kInvB], an[kInvB], bn[kInvB], cn[kInvB];
      // rows i0, i0 - 1, .. (those below 0 are not used)
      auto ld = [&](int32_t i0, double (&y)[kInvB], double (&u)[kInvB], double (&v)[kInvB],
                    double (&w)[kInvB]) {
        i0 = max(i0, kInvB - 1);
#pragma unroll
        for (int k = 0; k < kInvB; ++k) {
          y[k] = f[5][i0 - k];
          u[k] = f[0][i0 - k];
          v[k] = f[1][i0 - k];
          w[k] = f[2][i0 - k];
        }
      };
      auto run = [&](int32_t i0, const double (&y)[kInvB], const double (&u)[kInvB],
                     const double (&v)[kInvB], const double (&w)[kInvB]) {
#pragma unroll
        for (int k = 0; k < kInvB; ++k) {
          const double xi = (y[k] - v[k] * x1 - w[k] * x2) * u[k];
          f[5][i0 - k] = xi;
          x2 = x1;
          x1 = xi;
        }
      };
      // whole batches from the end, then the first rows one by one
      int32_t i0 = m - 1;
      if (i0 >= kInvB - 1) ld(i0, yb, ab, bb, cb);
      for (; i0 >= 2 * kInvB - 1; i0 -= 2 * kInvB) {
        ld(i0 - kInvB, yn, an, bn, cn);
        run(i0, yb, ab, bb, cb);
        ld(i0 - 2 * kInvB, yb, ab, bb, cb);
        run(i0 - kInvB, yn, an, bn, cn);
      }
      if (i0 >= kInvB - 1) {
        run(i0, yb, ab, bb, cb);
        i0 -= kInvB;
      }
      for (; i0 >= 0; --i0) {
        const double xi = (f[5][i0] - f[1][i0] * x1 - f[2][i0] * x2) * f[0][i0];
        f[5][i0] = xi;
        x2 = x1;
        x1 = xi;
      }
    }
    __syncthreads();
    for (int32_t i = tid; i < m; i += 256) {
      const double v = f[5][i];
      ss += v * v;
      x[c0 + i] = v;
    }
    __syncthreads();
  }
  ss = block_sum(ss, red);
  if (tid == 0) sinv = 1.0 / sqrt(ss);
  __syncthreads();
  for (int32_t i = tid; i < n; i += 256) x[i] *= sinv;
}

// Gram-Schmidt of at most kMaxVec normalised vectors against the earlier ones of the same
// cluster, in order, and normalisation; a vector without close ones stays as it is.
__global__ __launch_bounds__(256) void k_invit_gs(EigWs ws, int32_t n, int32_t nvec) {
  __shared__ double red[4];
  __shared__ double sinv;
  const double tnorm = ws.sc[S_TNORM];
  const int tid = threadIdx.x;
  for (int kv = 1; kv < nvec; ++kv) {
    double *x = ws.X + (int64_t)kv * n;
    const double lam = ws.eval[n - 1 - kv];
    bool any = false;
    for (int pv = 0; pv < kv; ++pv) {
      if (fabs(lam - ws.eval[n - 1 - pv]) > 1e-3 * tnorm) continue;
      any = true;
      const double *p = ws.X + (int64_t)pv * n;
      double s = 0.0;
      for (int32_t i = tid; i < n; i += 256) s += x[i] * p[i];
      s = block_sum(s, red);
      for (int32_t i = tid; i < n; i += 256) x[i] -= s * p[i];
      __syncthreads();
    }
    if (!any) continue;
    double s = 0.0;
    for (int32_t i = tid; i < n; i += 256) s += x[i] * x[i];
    s = block_sum(s, red);
    if (tid == 0) sinv = 1.0 / sqrt(s);
    __syncthreads();
    for (int32_t i = tid; i < n; i += 256) x[i] *= sinv;
    __syncthreads();
  }
}

// ---- more than kMaxVec vectors ----
// The vectors are orthogonalised after each of the two solves, batch by batch of kMaxVec:
// two solves in a row turn the vectors of a repeated eigenvalue towards
// the one nearest to their shifts, and what is left between them after that is rounding
// (residuals of 1e-11 of the norm; orthogonalised in between, a few ulps).

// Orthonormalisation of a batch of nb <= 64 vectors (X, vector v at X + v n) among
// themselves by its Gram matrix: X <- X R^-1 with G = R^T R (Cholesky), the same vectors
// as Gram-Schmidt in order.  Its error grows with the square of the batch's condition
// number, so the caller runs it twice.  Three launches on many blocks instead of 2,016
// dot products and updates in turn by one block (4 ms an iteration at n = 1,203; all three
// take 0.085).
constexpr int kGsRows = 64;
__global__ __launch_bounds__(256) void k_gs_gram(const double *__restrict__ X, int32_t n, int32_t nb,
                                                 double *__restrict__ part) {
  __shared__ double sx[kMaxVec][kGsRows + 1];
  const int t = threadIdx.x, r0 = blockIdx.x * kGsRows;
  for (int e = t; e < kMaxVec * kGsRows; e += 256) {
    const int v = e / kGsRows, i = e % kGsRows;
    sx[v][i] = (v < nb && r0 + i < n) ? X[(int64_t)v * n + r0 + i] : 0.0;
  }
  __syncthreads();
  // 16 apart, so that the 16 lanes of a row of products read different banks
  const int v0 = t >> 4, u0 = t & 15;
  double g[4][4] = {};
#pragma unroll 4
  for (int i = 0; i < kGsRows; ++i)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) g[a][b] += sx[v0 + 16 * a][i] * sx[u0 + 16 * b][i];
  double *out = part + (int64_t)blockIdx.x * kMaxVec * kMaxVec;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) out[(v0 + 16 * a) * kMaxVec + u0 + 16 * b] = g[a][b];
}
// Rinv (upper triangular, [u][v]) from the nblk partial Gram matrices, summed in order.
// A vector that depends on the earlier ones to rounding gets a pivot of at least 1e-30 of
// its square norm, so that the factor stays finite.
__global__ __launch_bounds__(1024) void k_gs_chol(const double *__restrict__ part, int32_t nblk,
                                                  int32_t nb, double *__restrict__ Rinv) {
  __shared__ double row[2][kMaxVec], mul[2][kMaxVec], d0[kMaxVec], d[kMaxVec];
  const int c = threadIdx.x & 63, q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // rows q, q + 16, .. of column c: of G right of the column being eliminated, of the
  // inverse up to it
  double x[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
  for (int32_t b = 0; b < nblk; ++b)
#pragma unroll
    for (int h = 0; h < 4; ++h) x[h] += part[((int64_t)b * kMaxVec + q + 16 * h) * kMaxVec + c];
#pragma unroll
  for (int h = 0; h < 4; ++h)
    if (c == q + 16 * h) d0[c] = x[h];
  // the owners (a wave) of row k leave it in LDS, and its multipliers: G stays symmetric, so
  // the row over the pivot is the column of multipliers too
  auto emit = [&](int k, double v) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), k);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), k);
    const double dk = fmax(__hiloint2double(hi, lo), 1e-30 * d0[k]);
    row[k & 1][c] = v;
    mul[k & 1][c] = v * rcp_nr(dk);
    if (c == 0) d[k] = dk;
  };
  __syncthreads();
  if (q == 0) emit(0, x[0]);
  __syncthreads();
  // elimination of [G | I] without square roots: step k changes the rows below k only, by
  // row k: one barrier a step (30 us at 19 parts; G and the inverse in LDS took 54, a
  // Cholesky factor and a back substitution 103)
  for (int k = 0; k < nb; ++k) {
    const double gc = row[k & 1][c];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int r = q + 16 * h;
      if (r > k) {
        const double m = mul[k & 1][r];
        x[h] = c == k ? -m : x[h] - m * gc;
        if (r == k + 1) emit(r, x[h]);
      }
    }
    __syncthreads();
  }
  // rows of the inverse over the pivots' roots are L^-1; R^-1 is its transpose
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int v = q + 16 * h;
    Rinv[c * kMaxVec + v] = (v < nb && c <= v) ? (c == v ? 1.0 : x[h]) / sqrt(d[v]) : 0.0;
  }
}
__global__ __launch_bounds__(256) void k_gs_apply(double *__restrict__ X, int32_t n, int32_t nb,
                                                  const double *__restrict__ Rinv) {
  __shared__ double sx[kMaxVec][kGsRows + 1], sr[kMaxVec][kMaxVec];
  const int t = threadIdx.x, r0 = blockIdx.x * kGsRows;
  for (int e = t; e < kMaxVec * kGsRows; e += 256) {
    const int v = e / kGsRows, i = e % kGsRows;
    sx[v][i] = (v < nb && r0 + i < n) ? X[(int64_t)v * n + r0 + i] : 0.0;
    sr[e / kMaxVec][e % kMaxVec] = Rinv[e];
  }
  __syncthreads();
  // 4 rows x 4 vectors a thread, rows 16 apart (different banks), vectors 16 apart
  const int i0 = t & 15, v0 = t >> 4;
  double y[4][4] = {};
#pragma unroll 4
  for (int u = 0; u < nb; ++u)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) y[a][b] += sx[u][i0 + 16 * a] * sr[u][v0 + 16 * b];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int i = i0 + 16 * a, v = v0 + 16 * b;
      if (v < nb && r0 + i < n) X[(int64_t)v * n + r0 + i] = y[a][b];
    }
}

// zeros in place of what the matrix held left of each reflector's first entry within its
// panel (rows c0 .. c0 + q of reflector q), so that a panel is a plain n x 32 operand
__global__ void k_bt_clean(EigWs ws, int32_t n, int32_t last) {
  const int32_t c = blockIdx.x * 8 + (threadIdx.x >> 5), i = threadIdx.x & 31;
  if (c > last) return;
  const int32_t c0 = c / kNB * kNB;
  if (c0 + i <= c) ws.a[(int64_t)c * ws.lda + c0 + i] = 0.0;
}

// ---------------------------------------------------------------- back-transform
// Panel p holds reflector rows c0 = p*kNB .. c0+nb-1 (v_q in A[c0+q][c0+q+1:],
// v_q[c0+q+1] = 1).  k_bt_gram forms G = V^T V over the panel's rows in kBtSplit
// row ranges (one block each, partial G into part1), k_bt_prep sums a panel's partials
// in range order and forms T (dlarft forward, columnwise:
// T[0:j, j] = -tau_j T[0:j, 0:j] G[0:j, j]) into Tall[p].  part1 holds
// (p_last + 1) * kBtSplit * kNB^2 doubles: 16 KNB^2 per 32 matrix rows, within its
// 512 doubles per row.
constexpr int kBtRows = 32;
constexpr int kBtSplit = 16;   // row ranges per panel in k_bt_gram
constexpr int kBtGRows = 128;  // rows staged per round in k_bt_gram
__device__ __forceinline__ int32_t bt_gram_rows(int32_t n, int32_t c0) {
  const int32_t rows = n - c0 - 1;  // reflector rows c0 + 1 .. n - 1
  return (rows + kBtSplit * kBtGRows - 1) / (kBtSplit * kBtGRows) * kBtGRows;
}
__global__ __launch_bounds__(256) void k_bt_gram(EigWs ws, int32_t n, int32_t last) {
  __shared__ double sv[kNB][kBtGRows + 1];
  const int32_t p = blockIdx.x, s = blockIdx.y;
  const int32_t c0 = p * kNB;
  const int32_t nb = min(kNB, last - c0 + 1);
  const int32_t per = bt_gram_rows(n, c0);
  const int32_t r_beg = c0 + 1 + s * per, r_end = min(n, r_beg + per);
  if (r_beg >= r_end) return;
  const int32_t lda = ws.lda;
  // element k of a thread: reflector q = (t + 256 k) / 128, row offset (t + 256 k) % 128;
  // indices are clamped so every load is unconditional, and masked when staged
  auto load = [&](int32_t rb, double (&v)[16]) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int idx = threadIdx.x + 256 * k, q = idx / kBtGRows, i = idx % kBtGRows;
      const int32_t cq = c0 + min(q, nb - 1), r = min(rb + i, n - 1);
      v[k] = ws.a[(int64_t)cq * lda + r];
    }
  };
  double g[4] = {0.0, 0.0, 0.0, 0.0}, cur[16], nxt[16];
  load(r_beg, cur);
  for (int32_t rb = r_beg; rb < r_end; rb += kBtGRows) {
    __syncthreads();  // the previous round's reads of sv are done
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int idx = threadIdx.x + 256 * k, q = idx / kBtGRows, i = idx % kBtGRows;
      const int32_t r = rb + i;
      sv[q][i] = (q < nb && r < r_end && r > c0 + q) ? cur[k] : 0.0;
    }
    __syncthreads();
    if (rb + kBtGRows < r_end) load(rb + kBtGRows, nxt);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int idx = threadIdx.x + 256 * k;
      const int q1 = idx / kNB, q2 = idx % kNB;
      double a = 0.0;
#pragma unroll 8
      for (int i = 0; i < kBtGRows; ++i) a += sv[q1][i] * sv[q2][i];
      g[k] += a;
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) cur[k] = nxt[k];
  }
  double *out = ws.part1 + ((int64_t)p * kBtSplit + s) * (kNB * kNB);
#pragma unroll
  for (int k = 0; k < 4; ++k) out[threadIdx.x + 256 * k] = g[k];
}
__global__ __launch_bounds__(256) void k_bt_prep(EigWs ws, int32_t n, int32_t last) {
  __shared__ double G[kNB][kNB + 1], tau[kNB];
  const int32_t p = blockIdx.x;
  const int32_t c0 = p * kNB;
  const int32_t nb = min(kNB, last - c0 + 1);
  const int32_t per = bt_gram_rows(n, c0);
  const int32_t nsp = (n - c0 - 1 + per - 1) / per;  // row ranges holding rows
  const double *src = ws.part1 + (int64_t)p * kBtSplit * (kNB * kNB);
  double g[4] = {0.0, 0.0, 0.0, 0.0};
  for (int32_t s = 0; s < nsp; ++s)
#pragma unroll
    for (int k = 0; k < 4; ++k) g[k] += src[(int64_t)s * (kNB * kNB) + threadIdx.x + 256 * k];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = threadIdx.x + 256 * k;
    G[idx / kNB][idx % kNB] = g[k];
  }
  if (threadIdx.x < kNB) tau[threadIdx.x] = (int)threadIdx.x < nb ? ws.tau[c0 + threadIdx.x] : 0.0;
  __syncthreads();
  if (threadIdx.x >= kNB) return;
  // a row of T needs only itself and G: a lane per row, no barriers (column by column with
  // the rows in LDS took 29 us, now 10)
  const int i = threadIdx.x;
  double row[kNB];
#pragma unroll
  for (int jj = 0; jj < kNB; ++jj) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < jj; ++k) s += row[k] * G[k][jj];
    row[jj] = i < jj ? -tau[jj] * s : (i == jj ? tau[jj] : 0.0);
  }
  double *T = ws.Tall + ((int64_t)p * kNB + i) * kNB;
#pragma unroll
  for (int jj = 0; jj < kNB; ++jj) T[jj] = row[jj];
}

// All panels for one vector (a block): no launch per panel and no sums between blocks.  A
// wave forms the dots of four reflectors, a thread two products of T, then the threads update
// a row each, whose reflector entries are loaded before the dots are known.  Bound by those
// two trips to L2 a panel and by what one block can read: with T, ten vectors of order 300
// take 0.086 ms (0.161 by k_bt_step and k_bt_reduce), 1,000 0.28 (0.39), 1,600 0.53 (0.60),
// 2,000 0.76 (0.75), where the line lies.
constexpr int kBtVecN = 1600;
__global__ __launch_bounds__(512) void k_bt_vec(EigWs ws, int32_t n, int32_t last) {
  constexpr int R = kNB / 8;  // reflectors per wave
  __shared__ double sx[kBtVecN], ss[kNB], sz[kNB];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int32_t lda = ws.lda;
  double *x = ws.X + (int64_t)blockIdx.x * n;
  for (int32_t i = t; i < n; i += 512) sx[i] = x[i];
  __syncthreads();
  for (int32_t p = last / kNB; p >= 0; --p) {
    const int32_t c0 = p * kNB, nb = min(kNB, last - c0 + 1);
    const double *T = ws.Tall + (int64_t)p * kNB * kNB + t;  // T_p[t / 32][t % 32] and 16 rows on
    const double t0 = T[0], t1 = T[512];
    const double *vq[R];
    double s[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      vq[u] = ws.a + (int64_t)(c0 + min(R * w + u, nb - 1)) * lda;
      s[u] = 0.0;
    }
#pragma unroll 4
    for (int32_t r = c0 + 1 + lane; r < n; r += 64) {
      const double xr = sx[r];
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const double a = vq[u][r];
        s[u] += (r > c0 + R * w + u ? a : 0.0) * xr;
      }
    }
    auto entries = [&](int32_t r, double (&v)[kNB]) {
      const int32_t at = min(r, n - 1);  // rows past the end read the last one
#pragma unroll
      for (int q = 0; q < kNB; ++q) v[q] = (ws.a + (int64_t)(c0 + min(q, nb - 1)) * lda)[at];
    };
    double v[kNB];
    int32_t r = c0 + 1 + t;
    entries(r, v);
#pragma unroll
    for (int u = 0; u < R; ++u) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s[u] += xlane(s[u], o);
      if (lane == 0) ss[R * w + u] = R * w + u < nb ? s[u] : 0.0;
    }
    __syncthreads();
    double z0 = t0 * ss[t & (kNB - 1)], z1 = t1 * ss[t & (kNB - 1)];
#pragma unroll
    for (int o = kNB / 2; o > 0; o >>= 1) {
      z0 += xlane(z0, o);
      z1 += xlane(z1, o);
    }
    if ((t & (kNB - 1)) == 0) {
      sz[t / kNB] = t / kNB < nb ? z0 : 0.0;
      sz[t / kNB + 16] = t / kNB + 16 < nb ? z1 : 0.0;
    }
    __syncthreads();
    for (;;) {
      double y = 0.0;
#pragma unroll
      for (int q = 0; q < kNB; ++q) y += (r > c0 + q ? v[q] : 0.0) * sz[q];
      if (r < n) sx[r] -= y;
      r += 512;
      if (r >= n) break;
      entries(r, v);
    }
    __syncthreads();
  }
  for (int32_t i = t; i < n; i += 512) x[i] = sx[i];
}

// Fused step for panel p: X[r] -= sum_q v_{p+1,q}[r] Z[q] (previous panel, if any),
// then this block's partial dots V_p^T X; k_bt_reduce forms Z <- T_p (V_p^T X).
__global__ __launch_bounds__(256) void k_bt_step(EigWs ws, int32_t n, int32_t p, int32_t last,
                                                 int32_t nvec, int32_t apply_prev) {
  __shared__ double szbuf[kNB * kMaxVec];
  __shared__ double sv[kNB][kBtRows + 1];   // this panel's reflectors over the block's rows
  __shared__ double svn[kNB][kBtRows + 1];  // the previous (higher) panel's
  __shared__ double sx[kMaxVec][kBtRows + 1];
  double(*sz)[kMaxVec] = (double(*)[kMaxVec])szbuf;
  const int32_t lda = ws.lda;
  const int32_t c0 = p * kNB;
  const int32_t nb = min(kNB, last - c0 + 1);
  const int32_t rbase = c0 + 1 + blockIdx.x * kBtRows;
  const int32_t rows = min(kBtRows, n - rbase);
  const int32_t c0n = c0 + kNB;  // previous (higher) panel
  const int32_t nbn = apply_prev ? min(kNB, last - c0n + 1) : 0;
  // every operand goes to LDS in one round of loads: Z, the block's rows of X, and
  // both panels' reflector entries over those rows.  All loads are issued before the
  // first LDS store (indices clamped into range; entries outside are stored as zero).
  constexpr int kZU = kNB * kMaxVec / 256, kXU = kMaxVec * kBtRows / 256;
  constexpr int kVU = kNB * kBtRows / 256;
  double zv[kZU], xv[kXU], vv[kVU], vnv[kVU] = {};
  const int t = threadIdx.x;
  if (apply_prev) {
#pragma unroll
    for (int u = 0; u < kZU; ++u) zv[u] = ws.Z[t + 256 * u];  // the whole kNB x kMaxVec block
  }
#pragma unroll
  for (int u = 0; u < kXU; ++u) {
    const int idx = t + 256 * u, o = min(idx / kBtRows, nvec - 1), i = min(idx % kBtRows, rows - 1);
    if (256 * u < nvec * kBtRows) xv[u] = ws.X[(int64_t)o * n + rbase + i];
  }
#pragma unroll
  for (int u = 0; u < kVU; ++u) {
    const int idx = t + 256 * u, q = idx / kBtRows, i = min(idx % kBtRows, rows - 1);
    vv[u] = ws.a[(int64_t)(c0 + min(q, nb - 1)) * lda + rbase + i];
    if (nbn > 0) vnv[u] = ws.a[(int64_t)(c0n + min(q, nbn - 1)) * lda + rbase + i];
  }
  __builtin_amdgcn_sched_barrier(0);
  if (apply_prev) {
#pragma unroll
    for (int u = 0; u < kZU; ++u) szbuf[t + 256 * u] = zv[u];
  }
#pragma unroll
  for (int u = 0; u < kXU; ++u) {
    const int idx = t + 256 * u, o = idx / kBtRows, i = idx % kBtRows;
    if (256 * u < nvec * kBtRows && o < nvec) sx[o][i] = i < rows ? xv[u] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < kVU; ++u) {
    const int idx = t + 256 * u, q = idx / kBtRows, i = idx % kBtRows;
    const int32_t r = rbase + i;
    sv[q][i] = (q < nb && i < rows && r > c0 + q) ? vv[u] : 0.0;
    svn[q][i] = (q < nbn && i < rows && r > c0n + q) ? vnv[u] : 0.0;
  }
  __syncthreads();
  if (apply_prev) {
    for (int idx = threadIdx.x; idx < nvec * kBtRows; idx += 256) {
      const int o = idx / kBtRows, i = idx % kBtRows;
      if (i >= rows) continue;
      double s = 0.0;
      for (int q = 0; q < nbn; ++q) s += svn[q][i] * sz[q][o];
      sx[o][i] -= s;
      ws.X[(int64_t)o * n + rbase + i] = sx[o][i];
    }
  }
  __syncthreads();  // sx updated
  // this block's partial dots V_p^T X over its rows; k_bt_reduce sums them
  const int nd = kNB * nvec;
  for (int idx = threadIdx.x; idx < nd; idx += 256) {
    const int q = idx / nvec, o = idx % nvec;
    double s = 0.0;
    for (int i = 0; i < rows; ++i) s += sv[q][i] * sx[o][i];
    ws.part1[(int64_t)blockIdx.x * nd + idx] = s;
  }
}

// Z_p = T_p (V_p^T X) from the partial dots of k_bt_step's nblk blocks: one block per
// vector o.  Thread (g, k) sums the partials
// b = g, g + 32, ... of entry (k, o), all its loads in one or two rounds; the 32 group
// sums are then added in group order and multiplied by T_p.
__global__ __launch_bounds__(1024) void k_bt_reduce(EigWs ws, int32_t p, int32_t last,
                                                    int32_t nvec, int32_t nblk) {
  __shared__ double acc[32][kNB + 1];
  __shared__ double col[kNB];
  __shared__ double sT[kNB][kNB + 1];
  const int o = blockIdx.x;
  const int nd = kNB * nvec;
  const int32_t nb = min(kNB, last - p * kNB + 1);
  const int k = threadIdx.x % kNB, g = threadIdx.x / kNB;
  const double tv = ws.Tall[(int64_t)p * kNB * kNB + threadIdx.x];  // T_p, one entry each
  acc[g][k] = sum_strided(ws.part1 + k * nvec + o, nd, g, 32, nblk);
  sT[g][k] = tv;
  __syncthreads();
  if (threadIdx.x < kNB) {
    double s = acc[0][k];
    for (int gg = 1; gg < 32; ++gg) s += acc[gg][k];
    col[k] = s;
  }
  __syncthreads();
  if (threadIdx.x < kNB) {
    const int q = threadIdx.x;
    double s = 0.0;
    for (int kk = q; kk < nb; ++kk) s += sT[q][kk] * col[kk];
    ws.Z[q * kMaxVec + o] = s;
  }
}

// final application of panel 0's Z
__global__ __launch_bounds__(256) void k_bt_apply0(EigWs ws, int32_t n, int32_t last,
                                                   int32_t nvec) {
  const int32_t r = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int32_t nb = min(kNB, last + 1);
  double v[kNB];
#pragma unroll
  for (int q = 0; q < kNB; ++q) v[q] = (q < nb && r > q) ? ws.a[(int64_t)q * ws.lda + r] : 0.0;
  for (int o = 0; o < nvec; ++o) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kNB; ++q) s += v[q] * ws.Z[q * kMaxVec + o];
    ws.X[(int64_t)o * n + r] -= s;
  }
}

// normalise + sign rule (largest |.| component positive, first on ties)
__global__ __launch_bounds__(256) void k_finish_vec(EigWs ws, int32_t n) {
  __shared__ double red[4];
  __shared__ double bv[256];
  __shared__ int32_t bi[256];
  __shared__ double fac;
  double *x = ws.X + (int64_t)blockIdx.x * n;
  double s = 0.0, best = -1.0;
  // start from an element this thread owns (or 0): the index stays in bounds even
  // when no comparison succeeds (a vector of NaNs)
  int32_t besti = (int32_t)threadIdx.x < n ? (int32_t)threadIdx.x : 0;
  for (int32_t i = threadIdx.x; i < n; i += 256) {
    s += x[i] * x[i];
    double a = fabs(x[i]);
    if (a > best) {
      best = a;
      besti = i;
    }
  }
  s = block_sum(s, red);
  bv[threadIdx.x] = best;
  bi[threadIdx.x] = besti;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      double b2 = bv[threadIdx.x + o];
      int32_t i2 = bi[threadIdx.x + o];
      if (b2 > bv[threadIdx.x] || (b2 == bv[threadIdx.x] && i2 < bi[threadIdx.x])) {
        bv[threadIdx.x] = b2;
        bi[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double f = 1.0 / sqrt(s);
    const int32_t ib = bi[0];
    if (ib >= 0 && ib < n && x[ib] < 0.0) f = -f;
    fac = f;
  }
  __syncthreads();
  for (int32_t i = threadIdx.x; i < n; i += 256) x[i] *= fac;
}

// ---------------------------------------------------------------- driver
static void launch_tridiag(EigWs ws, int32_t n, int32_t stop, hipStream_t st) {
  hipLaunchKernelGGL(k_col0, dim3(1), dim3(256), 0, st, ws, n);
  for (int32_t c = 0; c + 1 < n && c < stop; ++c) {
    const int32_t j = c % kNB;
    const int32_t L = n - c - 1;
    const int32_t gs = symv_tiles(n, c), gw = (L + kWRows - 1) / kWRows;
    hipLaunchKernelGGL(k_symv, dim3((unsigned)gs), dim3(256), 0, st, ws, n, c, j);
    hipLaunchKernelGGL(k_wcol, dim3((unsigned)gw), dim3(256), 0, st, ws, n, c, j, gs);
    // panel end: update the trailing matrix before the next panel's first symv
    if (j == kNB - 1 && c + 2 < n) {
      const int32_t k1 = c + 1;
      const int32_t nt = (n - k1 + 63) / 64;
      hipLaunchKernelGGL(k_syr2k, dim3((unsigned)(nt * (nt + 1) / 2)), dim3(256), 0, st, ws, n, k1,
                         kNB);
    }
  }
}

// ---- the resident part's launch shapes: the order a shape holds, and its kernel.  A stage
// runs the smallest shape that holds what is left, down to the next smaller one's order:
// a column costs an exchange (about 1.7 us) and the work between, which grows with the
// blocks and the columns per thread.  Measured, whole reductions: n = 198 0.46 ms, 512
// 1.27, 1,000 2.66, 2,048 7.1, where launches per column took 1.5, 4.9, 9.6 and 22.  n =
// 1,000 in the 1,024 shape alone takes 0.3 ms longer than by stages.  Above 2,048 the rows
// and the four vectors no longer fit 256 registers a thread: 512 x 6 columns x 12 rows
// spills and takes 18 to 29 us a column, more than the launches.
struct TriShape {
  int32_t cap, T, RS;
  void (*fn)(EigWs, int32_t, int32_t, int32_t, double *, double *, int64_t);
};
static const TriShape kTriShapes[] = {
    {256, 256, 8, k_tri<256, 1, 8>},   {512, 256, 8, k_tri<256, 2, 8>},
    {1024, 512, 8, k_tri<512, 2, 8>},  {2048, 512, 8, k_tri<512, 4, 8>},
};
constexpr int kTriNum = sizeof(kTriShapes) / sizeof(kTriShapes[0]);
// one resident launch at a time on a device (see k_tri)
static std::mutex g_tri_mu[16];

// largest order that a launch of blocks one per CU holds, at most `cap`
static int32_t tri_cap(const eig_ctx *ctx) {
  int32_t best = 0;
  for (const TriShape &h : kTriShapes)
    if ((h.cap + h.RS - 1) / h.RS <= ctx->num_cu) best = std::max(best, h.cap);
  return best;
}
static int launch_resident(eig_ctx *ctx, const EigWs &ws, int32_t n, int32_t c0, hipStream_t st) {
  // exchange buffers: products and rows, one word per column and row of a stage
  auto stage = [&](int32_t c, int32_t &c1) -> const TriShape * {
    int i = 0;
    while (kTriShapes[i].cap < n - c) ++i;
    c1 = i == 0 ? n - 1 : std::min(n - 1, n - kTriShapes[i - 1].cap);
    return &kTriShapes[i];
  };
  int64_t words = 0;
  for (int32_t c = c0, c1; c < n - 1; c = c1) {
    stage(c, c1);
    words = std::max(words, (int64_t)(c1 - c) * (n - c));
  }
  EIG_TRY(eig_ensure(ctx, ctx->tribuf, 16 * (size_t)words));
  double *yb = (double *)ctx->tribuf.p;
  for (int32_t c = c0, c1; c < n - 1; c = c1) {
    const TriShape *h = stage(c, c1);
    const int64_t ld = n - c, cnt = 2 * (int64_t)(c1 - c) * ld;
    hipLaunchKernelGGL(k_tri_fill, dim3((unsigned)std::min<int64_t>((cnt + 255) / 256, 4096)), dim3(256), 0,
                       st, (uint64_t *)yb, cnt);
    hipLaunchKernelGGL(h->fn, dim3((unsigned)((n - c + h->RS - 1) / h->RS)), dim3((unsigned)h->T), 0, st, ws,
                       n, c, c1, yb, yb + (int64_t)(c1 - c) * ld, ld);
  }
  EIG_HIP(ctx, hipGetLastError());
  return EIG_OK;
}

static int run_eigh(eig_ctx *ctx, const double *d_a, int32_t n, int32_t nvec, double *evals,
                    double *evecs, bool internal, bool resident, bool *again);

int eig_run_eigh(eig_ctx *ctx, const double *d_a, int32_t n, int32_t nvec, double *evals,
                 double *evecs, bool internal) {
  EigInUse busy(ctx->in_eigh);
  bool again = false;
  EIG_TRY(run_eigh(ctx, d_a, n, nvec, evals, evecs, internal, true, &again));
  // the resident part gave up waiting for blocks that were not scheduled: start over with
  // the launches that wait for nothing outside themselves
  if (again) EIG_TRY(run_eigh(ctx, d_a, n, nvec, evals, evecs, internal, false, &again));
  return EIG_OK;
}

static int run_eigh(eig_ctx *ctx, const double *d_a, int32_t n, int32_t nvec, double *evals,
                    double *evecs, bool internal, bool resident, bool *again) {
  *again = false;
  if (n <= 0) return eig_set_err(ctx, EIG_E_ARG, "eigh: n <= 0");
  if (nvec < 0 || nvec > n) return eig_set_err(ctx, EIG_E_ARG, "eigh: nvec must be in [0, n]");
  if (internal && nvec > kMaxVec)
    return eig_set_err(ctx, EIG_E_ARG, "eigh: internal calls take at most %d vectors", kMaxVec);
  // an internal call leaves the caller's stage timing (same events) running
  auto tbeg = [&]() { if (!internal) eig_time_begin(ctx); };
  auto tend = [&](const char *what) { if (!internal) eig_time_end(ctx, what); };
  const int64_t N = n;
  const int32_t lda = (int32_t)(((N + 7) / 8) * 8);
  const int64_t maxblk = (N + 3) / 4 + 8, ntile = (N + kSyT - 1) / kSyT;
  const int64_t maxnv = (int64_t)kNB * kMaxVec;
  const int64_t maxw = (N + kWRows - 1) / kWRows + 2;
  const int64_t npanel = (N + kNB - 1) / kNB + 1;
  size_t need = 0;
  auto add = [&](size_t cnt) {
    size_t o = need;
    need += ((cnt * 8 + 255) / 256) * 256;
    return o;
  };
  size_t o_a = add((size_t)N * lda);
  // cleared before a solve, one range
  size_t o_sc = add(S_COUNT), o_e = add(N), o_e2 = add(N), o_tau = add(N), o_V = add(kNB * N),
         o_W = add(kNB * N), o_x = add(lda), o_sync = add(8);
  size_t o_d = add(N), o_y = add((size_t)ntile * lda), o_p1 = add((size_t)maxblk * maxnv),
         o_ev = add(N), o_st = add(2 * (size_t)(sturm_rows(n) + kStB)),
         o_X = add((size_t)kMaxVec * N), o_lu = add((size_t)kMaxVec * kLuF * N),
         o_Z = add(kNB * kMaxVec), o_T = add((size_t)npanel * kNB * kNB),
         o_pw = add((size_t)2 * maxw * kPW), o_ps = add((size_t)(ntile * (ntile + 1) / 2));
  EIG_TRY(eig_ensure(ctx, ctx->ework, need));
  char *base = (char *)ctx->ework.p;
  EigWs ws;
  ws.a = (double *)(base + o_a);
  ws.lda = lda;
  ws.d = (double *)(base + o_d);
  ws.e = (double *)(base + o_e);
  ws.e2 = (double *)(base + o_e2);
  ws.tau = (double *)(base + o_tau);
  ws.V = (double *)(base + o_V);
  ws.W = (double *)(base + o_W);
  ws.xtmp = (double *)(base + o_x);
  ws.yp = (double *)(base + o_y);
  ws.sc = (double *)(base + o_sc);
  ws.part1 = (double *)(base + o_p1);
  ws.eval = (double *)(base + o_ev);
  ws.st = (double2 *)(base + o_st);
  ws.X = (double *)(base + o_X);
  ws.lu = (double *)(base + o_lu);
  ws.Z = (double *)(base + o_Z);
  ws.Tall = (double *)(base + o_T);
  ws.pw = (double *)(base + o_pw);
  ws.ps = (double *)(base + o_ps);
  ws.sync = (int32_t *)(base + o_sync);
  ws.maxw = (int32_t)maxw;
  hipStream_t st = ctx->stream;
  if (lda != n) EIG_HIP(ctx, hipMemsetAsync(ws.a, 0, sizeof(double) * N * lda, st));
  EIG_HIP(ctx, hipMemcpy2DAsync(ws.a, sizeof(double) * lda, d_a, sizeof(double) * N,
                                sizeof(double) * N, N, hipMemcpyDeviceToDevice, st));
  EIG_HIP(ctx, hipMemsetAsync(base + o_sc, 0, o_d - o_sc, st));

  // ---- tridiagonalisation: plain launches.  The host queues a launch in ~3 us, less than
  // the shortest column takes on the device, so a captured graph of the launches replays
  // no faster (n = 5,000: 97.5 against 96.4 ms) and capturing it costs every first solve of
  // an order or a context 12.5 ms.
  tbeg();
  // long columns by launches, whole panels, until the resident part holds the rest.
  // EIG_NO_MERGE=1 runs all columns by launches: counter-collection runs use it, since no
  // launch then waits on other blocks of its own grid
  const int32_t cap = resident && getenv("EIG_NO_MERGE") == nullptr ? tri_cap(ctx) : 0;
  const int32_t stop = cap == 0 ? n : (n > cap ? (n - cap + kNB - 1) / kNB * kNB : 0);
  if (stop > 0) launch_tridiag(ws, n, stop, st);
  EIG_HIP(ctx, hipGetLastError());
  if (stop < n - 1) {
    std::lock_guard<std::mutex> lock(g_tri_mu[ctx->device & 15]);
    EIG_TRY(launch_resident(ctx, ws, n, stop, st));
    int32_t gave_up[2] = {0, 0};
    EIG_HIP(ctx, hipMemcpyAsync(gave_up, ws.sync, sizeof(gave_up), hipMemcpyDeviceToHost, st));
    EIG_HIP(ctx, hipStreamSynchronize(st));
    if (gave_up[1] == 2) {
      *again = true;
      return EIG_OK;
    }
  } else if (n == 1) {
    hipLaunchKernelGGL(k_col0, dim3(1), dim3(256), 0, st, ws, n);
  }
  tend("tridiag");
  // ---- eigenvalues
  tbeg();
  hipLaunchKernelGGL(k_gersh, dim3(1), dim3(256), 0, st, ws, n);
  hipLaunchKernelGGL(k_sturm_prep, dim3((unsigned)((sturm_rows(n) + kStB + 255) / 256)), dim3(256), 0, st, ws, n);
  {
    // the grid's counts go to the inverse iteration's LU area, unused until then
    // (kMaxVec * 5 * N doubles hold the kMsGrid counts from N = 103 on)
    int32_t *gcnt = nullptr;
    if ((int64_t)kMaxVec * kLuF * N * 2 >= kMsGrid && n >= 128) {
      gcnt = (int32_t *)ws.lu;
      hipLaunchKernelGGL(k_msgrid, dim3(kMsGrid / 256), dim3(256), 0, st, ws, n, gcnt);
    }
    int32_t lanes = 64;
    while (lanes > 8 && (int64_t)n * lanes > (int64_t)ctx->num_cu * 256) lanes /= 2;
    auto kern = lanes == 64   ? k_multisect<64>
                : lanes == 32 ? k_multisect<32>
                : lanes == 16 ? k_multisect<16>
                              : k_multisect<8>;
    hipLaunchKernelGGL(kern, dim3((unsigned)(((int64_t)n * lanes + 255) / 256)), dim3(256), 0, st, ws, n,
                       (const int32_t *)gcnt);
  }
  EIG_HIP(ctx, hipGetLastError());
  tend("bisect");
  // ---- eigenvectors: one batch of at most kMaxVec (inverse iteration with Gram-Schmidt,
  // back-transform, sign rule); more vectors run in batches of kMaxVec in eigenvalue
  // order: twice every batch's solve and batch by batch the Gram-Schmidt against the earlier
  // vectors and within the batch, then the back-transform of all
  // vectors together as FP64 MFMA products
  const int32_t last = n - 2;  // last reflector row
  const int32_t p_last = last >= 0 ? last / kNB : -1;
  auto back_transform = [&](int32_t nb) -> int {
    if (last >= 0 && n <= kBtVecN) {
      hipLaunchKernelGGL(k_bt_vec, dim3((unsigned)nb), dim3(512), 0, st, ws, n, last);
    } else if (last >= 0) {
      for (int32_t p = p_last; p >= 0; --p) {
        const int32_t c0 = p * kNB;
        const unsigned g = (unsigned)((n - c0 - 1 + kBtRows - 1) / kBtRows);
        hipLaunchKernelGGL(k_bt_step, dim3(g), dim3(256), 0, st, ws, n, p, last, nb,
                           (int32_t)(p < p_last));
        hipLaunchKernelGGL(k_bt_reduce, dim3((unsigned)nb), dim3(1024), 0, st, ws, p, last, nb,
                           (int32_t)g);
      }
      hipLaunchKernelGGL(k_bt_apply0, dim3((unsigned)((n - 1 + 255) / 256)), dim3(256), 0, st, ws,
                         n, last, nb);
    }
    hipLaunchKernelGGL(k_finish_vec, dim3((unsigned)nb), dim3(256), 0, st, ws, n);
    EIG_HIP(ctx, hipGetLastError());
    return EIG_OK;
  };
  tbeg();
  if (nvec > 0 && nvec <= kMaxVec) {
    // two iterations: the eigenvalues are accurate to a few ulps, so one solve already
    // leaves contamination of order eps ||T|| / gap from outside a cluster, and the
    // second squares it (the parity tests pass with one; two keep a margin)
    for (int it = 0; it < 2; ++it) {
      hipLaunchKernelGGL(k_invit_solve, dim3((unsigned)nvec), dim3(256), 0, st, ws, n, 0, (int32_t)(it == 0),
                         (int32_t)(it == 0), ws.X, ws.lu);
      hipLaunchKernelGGL(k_invit_gs, dim3(1), dim3(256), 0, st, ws, n, nvec);
    }
    tend("invit");
    tbeg();
    if (last >= 0) {
      hipLaunchKernelGGL(k_bt_gram, dim3((unsigned)(p_last + 1), kBtSplit), dim3(256), 0, st, ws, n,
                         last);
      hipLaunchKernelGGL(k_bt_prep, dim3((unsigned)(p_last + 1)), dim3(256), 0, st, ws, n, last);
    }
    EIG_TRY(back_transform(nvec));
  } else if (nvec > kMaxVec) {
    // all vectors (vector j at j N), the Gram-Schmidt and back-transform coefficients, the
    // partial Gram matrices, R^-1, and the LU factors of as many vectors as 2 GiB hold
    const int32_t nblk = (n + kGsRows - 1) / kGsRows;
    const size_t lub = (size_t)kLuF * N;
    const int32_t group = (int32_t)std::max<size_t>(1, std::min<size_t>(nvec, ((size_t)1 << 28) / lub));
    const size_t sq = (size_t)kMaxVec * kMaxVec;
    const size_t kpart = (size_t)8 * kMaxVec * N;  // the parts of products over a long k
    EIG_TRY(eig_ensure(ctx, ctx->evall, sizeof(double) * ((size_t)N * nvec + (size_t)kMaxVec * nvec +
                                                          sq * nblk + sq + lub * group + kpart)));
    double *XT = (double *)ctx->evall.p, *Cc = XT + (size_t)N * nvec, *gp = Cc + (size_t)kMaxVec * nvec,
           *Ri = gp + sq * nblk, *lu = Ri + sq, *kp = lu + lub * group;
    // against every earlier vector, not only those of close eigenvalues: the products are
    // a small part, and vectors a few 1e-3 ||T|| apart stay orthogonal to the last ulps.
    // After the first solve once is enough (the vectors only start the second)
    for (int it = 0; it < 2; ++it) {
      for (int32_t b = 0; b < nvec; b += group)
        hipLaunchKernelGGL(k_invit_solve, dim3((unsigned)std::min(group, nvec - b)), dim3(256), 0, st, ws, n,
                           b, (int32_t)(it == 0), (int32_t)(it == 0 || nvec > group), XT, lu);
      EIG_HIP(ctx, hipGetLastError());
      for (int32_t j0 = 0; j0 < nvec; j0 += kMaxVec) {
        const int32_t nb = std::min<int32_t>(kMaxVec, nvec - j0), nc = j0;
        double *X = XT + (size_t)j0 * N;
        const double *P = XT;
        for (int rep = 0; rep <= it; ++rep) {
          if (nc > 0) {
            EIG_TRY(eig_gemm_f64_long(ctx, st, true, false, nc, nb, N, 1.0, P, N, X, N, 0.0, Cc, nc, false,
                                      kp, kpart));
            EIG_TRY(eig_gemm_f64_long(ctx, st, false, false, N, nb, nc, -1.0, P, N, Cc, nc, 1.0, X, N,
                                      false, kp, kpart));
          }
          hipLaunchKernelGGL(k_gs_gram, dim3((unsigned)nblk), dim3(256), 0, st, (const double *)X, n, nb, gp);
          hipLaunchKernelGGL(k_gs_chol, dim3(1), dim3(1024), 0, st, (const double *)gp, nblk, nb, Ri);
          hipLaunchKernelGGL(k_gs_apply, dim3((unsigned)nblk), dim3(256), 0, st, X, n, nb, (const double *)Ri);
        }
      }
    }
    EIG_HIP(ctx, hipGetLastError());
    tend("invit");
    tbeg();
    if (last >= 0) {
      hipLaunchKernelGGL(k_bt_gram, dim3((unsigned)(p_last + 1), kBtSplit), dim3(256), 0, st, ws, n,
                         last);
      hipLaunchKernelGGL(k_bt_prep, dim3((unsigned)(p_last + 1)), dim3(256), 0, st, ws, n, last);
      hipLaunchKernelGGL(k_bt_clean, dim3((unsigned)(last / 8 + 1)), dim3(256), 0, st, ws, n, last);
      double *Z = Cc + (size_t)kNB * nvec;
      for (int32_t p = p_last; p >= 0; --p) {
        const int32_t c0 = p * kNB, np = std::min(kNB, last - c0 + 1);
        const int64_t rows = N - c0 - 1;
        const double *Vp = ws.a + (size_t)c0 * lda + c0 + 1;
        EIG_TRY(eig_gemm_f64_long(ctx, st, true, false, np, nvec, rows, 1.0, Vp, lda, XT + c0 + 1, N,
                                  0.0, Cc, kNB, false, kp, kpart));
        EIG_TRY(eig_gemm_f64(ctx, st, true, false, np, nvec, np, 1.0, ws.Tall + (size_t)p * kNB * kNB,
                             kNB, 0, Cc, kNB, 0, 0.0, Z, kNB, 0, 1));
        EIG_TRY(eig_gemm_f64(ctx, st, false, false, rows, nvec, np, -1.0, Vp, lda, 0, Z, kNB, 0, 1.0,
                             XT + c0 + 1, N, 0, 1));
      }
    }
    EigWs wx = ws;
    wx.X = XT;
    hipLaunchKernelGGL(k_finish_vec, dim3((unsigned)nvec), dim3(256), 0, st, wx, n);
    EIG_HIP(ctx, hipGetLastError());
    if (!internal) {
      EIG_TRY(eig_ensure(ctx, ctx->evecs_dev, sizeof(double) * N * kMaxVec));
      EIG_HIP(ctx, hipMemcpyAsync(ctx->evecs_dev.p, XT, sizeof(double) * N * kMaxVec,
                                  hipMemcpyDeviceToDevice, st));
    }
  } else {
    tend("invit");
    tbeg();
  }
  tend("eigvec");
  std::vector<double> asc(N);
  EigFetch f(ctx);
  EIG_TRY(f.get(asc.data(), ws.eval, sizeof(double) * N));
  if (nvec > 0 && evecs)
    EIG_TRY(f.get(evecs, nvec <= kMaxVec ? ws.X : (double *)ctx->evall.p, sizeof(double) * N * nvec));
  if (nvec > 0 && nvec <= kMaxVec && !internal) {
    EIG_TRY(eig_ensure(ctx, ctx->evecs_dev, sizeof(double) * N * nvec));
    EIG_HIP(ctx, hipMemcpyAsync(ctx->evecs_dev.p, ws.X, sizeof(double) * N * nvec,
                                hipMemcpyDeviceToDevice, st));
  }
  EIG_TRY(f.wait());
  for (int64_t i = 0; i < N; ++i) {
    if (std::isnan(asc[i])) return eig_set_err(ctx, EIG_E_CONVERGE, "eigenvalue is NaN");
    if (evals) evals[i] = asc[N - 1 - i];
  }
  if (nvec > 0 && evecs)
    for (int64_t i = 0; i < N * nvec; ++i)
      if (!std::isfinite(evecs[i]))
        return eig_set_err(ctx, EIG_E_CONVERGE, "eigenvector %lld is not finite",
                           (long long)(i / N));
  if (!internal) ctx->last_nvec = nvec;
  return EIG_OK;
}

extern "C" int eig_eigh_xtx(eig_ctx *ctx, int32_t nvec, double *evals, double *evecs) {
  if (!ctx) return EIG_E_ARG;
  if (!ctx->have_xtx) return eig_set_err(ctx, EIG_E_STATE, "eig_eigh_xtx before eig_xtx");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  return eig_run_eigh(ctx, (const double *)ctx->xtx.p, ctx->nrows, nvec, evals, evecs);
}

extern "C" int eig_eigh(eig_ctx *ctx, const double *a, int32_t n, int32_t nvec, double *evals,
                        double *evecs) {
  if (!ctx || !a || n <= 0) return eig_set_err(ctx, EIG_E_ARG, "eig_eigh: args");
  for (int64_t i = 0; i < (int64_t)n * n; ++i)
    if (!std::isfinite(a[i])) return eig_set_err(ctx, EIG_E_ARG, "eig_eigh: matrix is not finite");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  EIG_TRY(eig_ensure(ctx, ctx->scratch, sizeof(double) * (size_t)n * n));
  EIG_HIP(ctx, hipMemcpyAsync(ctx->scratch.p, a, sizeof(double) * (size_t)n * n,
                              hipMemcpyHostToDevice, ctx->stream));
  return eig_run_eigh(ctx, (const double *)ctx->scratch.p, n, nvec, evals, evecs);
}
