// Launch plans and the sizes of the work areas they need: host arithmetic alone (no HIP), so
// that what a kernel will write can be checked against what is allocated without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

// ---- products of packed codes with FP64 columns (codes.hip)
constexpr int kCdDig = 7;        // digits per column
constexpr int kCdStage = 128;    // k per stage
constexpr int kCdFrag = 1024;    // bytes of a digit operand: 16 digit columns x 64 k
constexpr int kCdMaxCols = 20;   // columns of a group of nine tiles (140 of 144 digit columns)
constexpr int kCdMaxNT = 9;

enum { kCdPair, kCdSum, kCdMiss };
// Terms that one INT32 sum holds.  A term is a digit (-128 .. 127) times a code of up to 3, and
// with kCdSum, whose two planes meet in one sum, the missing bit's digit on top: 384 and 512.
constexpr int64_t cd_max_k(int mode) { return mode == kCdSum ? (int64_t)4 << 20 : (int64_t)5 << 20; }
static_assert(128 * 4 * cd_max_k(kCdSum) <= (int64_t)1 << 31 && 128 * 3 * cd_max_k(kCdPair) < (int64_t)1 << 31, "");
struct CodesPlan {
  int mode;
  int32_t C, ngroup, Cg, NT, R, nrowblk, nsplit;
  int64_t nblk, per, rowpad;
  size_t head_bytes, dig_bytes, part_bytes;
};

// row tiles of 16 per wave at most (a block is four waves)
constexpr int cd_tiles(int mode, int NT) {
  return mode == kCdPair ? 2 : mode == kCdSum && NT == kCdMaxNT ? 3 : 4;
}

// column groups: at most 20 columns (nine tiles), or 11 (five) when that is all
inline void cd_groups(int32_t C, int32_t &ngroup, int32_t &Cg, int32_t &NT) {
  ngroup = (C + kCdMaxCols - 1) / kCdMaxCols;
  Cg = (C + ngroup - 1) / ngroup;
  NT = Cg * kCdDig <= 80 ? 5 : 9;
}

// The product of nrow rows of codes with C columns over nblk stages, in at most smax splits
// (more only where an INT32 sum would not hold a split).
inline CodesPlan eig_codes_plan(int num_cu, int mode, int32_t C, int64_t nrow, int64_t nblk, int32_t smax) {
  CodesPlan P;
  P.mode = mode;
  P.C = C;
  P.nblk = nblk;
  cd_groups(C, P.ngroup, P.Cg, P.NT);
  // fewer row tiles a wave where the rows fill no more (three run as the most)
  P.R = (int32_t)std::min<int64_t>(cd_tiles(mode, P.NT), (nrow + 63) / 64);
  if (P.R > 2) P.R = cd_tiles(mode, P.NT);
  const int32_t rows = 64 * P.R;
  P.nrowblk = (int32_t)((nrow + rows - 1) / rows);
  P.rowpad = (int64_t)P.nrowblk * rows;
  // splits: rounds of the blocks the chip holds (two per CU) times stages each, plus the
  // sums' way to memory and back, worth about two stages a block
  const int64_t slots = 2 * (int64_t)std::max(num_cu, 1);
  const int64_t pmax = cd_max_k(mode) / kCdStage;  // stages of one INT32 sum
  const int64_t smin = (nblk + pmax - 1) / pmax;
  double best = 0.0;
  P.nsplit = 1;
  P.per = nblk;
  for (int64_t s = smin; s <= std::min<int64_t>(nblk, std::max<int64_t>(smax, smin)); ++s) {
    const int64_t pe = (nblk + s - 1) / s;
    if ((nblk + pe - 1) / pe != s) continue;
    const double rounds = (double)(((int64_t)P.nrowblk * P.ngroup * s + slots - 1) / slots);
    const double cost = rounds * ((double)pe + 2.0) + 1.0 * (double)P.nrowblk * P.ngroup * (double)s / (double)slots;
    if (best == 0.0 || cost < best) {
      best = cost;
      P.nsplit = (int32_t)s;
      P.per = pe;
    }
  }
  const int32_t planes = mode == kCdSum ? 2 : 1, nacc = mode == kCdPair ? 2 : 1;
  P.head_bytes = ((size_t)C * 24 + 255) / 256 * 256;
  P.dig_bytes = (size_t)P.ngroup * nblk * planes * P.NT * 2 * kCdFrag;
  P.part_bytes = (size_t)P.ngroup * P.nsplit * nacc * P.rowpad * P.NT * 16 * 4;
  return P;
}
// Where the regrouped codes of all SNPs (a copy of the selection) find no room, the products
// over SNPs take this many stages of them at a time: a sixteenth, from 16 MiB to 1 GiB.
inline int64_t eig_codes_chunk(int32_t nst, int64_t nblk) {
  const int64_t stage = (int64_t)nst * 4096;
  const int64_t b = std::min<int64_t>((int64_t)1 << 30, std::max<int64_t>((int64_t)16 << 20, stage * nblk / 16));
  return std::max<int64_t>(1, std::min(nblk, b / stage));
}
// a plan's scales, digit operands (a multiple of 2 KB) and INT32 sums, one after the other
inline size_t eig_codes_area(const CodesPlan &P) { return P.head_bytes + P.dig_bytes + P.part_bytes; }

// ---- fastmode's FP64 panel products (fpca.hip): X A and X^T B of the power iterations, and
// the finishing X^T U of a basis of r columns.  The digits of the products over SNPs and the
// sums of X A grow with the SNPs (3.1 and 1.2 KB each, with 20 and 220 columns): a pass takes
// as many SNPs as 4 GiB of either hold, which is all of them up to 1.4 and 3.7 million.
constexpr int64_t kFpcaBytes = (int64_t)4 << 30;
inline CodesPlan eig_fpca_plan(int num_cu, int mode, int32_t C, int64_t nrow, int64_t nblk) {
  CodesPlan one = eig_codes_plan(num_cu, mode, C, nrow, 1, 1);
  if (mode == kCdSum) {
    nblk = std::min<int64_t>(nblk, kFpcaBytes / (int64_t)one.dig_bytes);
  } else {
    const int64_t row = (int64_t)one.part_bytes / one.rowpad;
    nrow = std::min<int64_t>(nrow, kFpcaBytes / row / 128 * 128);
  }
  // splits whose sums stay within 2 GiB
  one = eig_codes_plan(num_cu, mode, C, nrow, nblk, 1);
  const size_t b = one.part_bytes / (size_t)one.nsplit;
  return eig_codes_plan(num_cu, mode, C, nrow, nblk,
                        (int32_t)std::max<size_t>(1, std::min<size_t>(32, ((size_t)2 << 30) / b)));
}
struct FpcaPlans {
  CodesPlan pa, pb;
  int64_t arows;  // SNPs of a pass of X A
  size_t area;    // holds each of them and the finishing product at every rank the basis may have
};
inline CodesPlan eig_fpca_basis_plan(int num_cu, int64_t M, int32_t nst, int32_t r) {
  return eig_fpca_plan(num_cu, kCdSum, r, (int64_t)nst * 128, (M + 127) / 128);
}
inline FpcaPlans eig_fpca_plans(int num_cu, int64_t M, int32_t nst, int32_t K, int32_t L, int32_t Ctot) {
  FpcaPlans F;
  F.pa = eig_fpca_plan(num_cu, kCdPair, L, M, nst);
  F.arows = std::min<int64_t>(M, F.pa.rowpad);
  F.pb = eig_fpca_plan(num_cu, kCdSum, L, (int64_t)nst * 128, (M + 127) / 128);
  F.area = std::max(eig_codes_area(F.pa), eig_codes_area(F.pb));
  // fewer columns can need more: their groups, and with them the row padding and the splits,
  // are chosen anew
  for (int32_t r = K; r <= Ctot; ++r)
    F.area = std::max(F.area, eig_codes_area(eig_fpca_basis_plan(num_cu, M, nst, r)));
  return F;
}

// ---- the FP64 XTX on digit planes (xdigit.hip)
constexpr int kXT = 256;          // samples per tile side
constexpr int kResSnps = 128;     // SNPs a step of the left-out parts' sums
constexpr int64_t kXMaxK = 131072;  // SNPs of one INT32 sum: 128 * (126 + 1) * 2^17 < 2^31
// Workspace that stays with the context: 8 GiB of planes (SNP chunks; 5,000 samples fill it at
// 600,000 SNPs) and 4 GiB of INT32 sums.  The sums of every tile pair at once are 1.4 GiB at
// 5,000 samples, 28 at 46,000 and 117 GB at 85,000, which would leave the eigensolver no
// room; past 4 GiB (2,340 pairs of 16,384 blocks, 64 rounds of the chip) the pairs run in bands.
constexpr int64_t kXPlaneBytes = (int64_t)8 << 30, kXPartBytes = (int64_t)4 << 30;
struct XdPlan {
  int32_t nT, RT, npair, np;  // tiles of kXT, row tiles of 32, tile pairs, planes
  int64_t K, nchunk;          // SNPs per chunk (a multiple of 128), chunks
  int32_t nsplit, per;        // splits of a chunk, 64-SNP stages each (even)
  int32_t band;               // tile pairs per pass
  int32_t rsplit, rstep;      // splits of the left-out parts' sums, steps of kResSnps in each
  size_t plane_bytes, tab_bytes, part_bytes;
};
// p1 and p2 digits of the two brackets
inline XdPlan eig_xd_plan(int num_cu, int64_t M, int32_t nst, int32_t p1, int32_t p2) {
  XdPlan X;
  X.nT = (nst + 1) / 2;
  X.RT = 8 * X.nT;
  X.npair = X.nT * (X.nT + 1) / 2;
  X.np = p1 + p2 + 2;
  const int64_t rows = (int64_t)X.RT * 32;
  const int64_t kmem = std::max<int64_t>(4096, kXPlaneBytes / (rows * X.np) / 128 * 128);
  const int64_t kmax = std::min<int64_t>(kXMaxK, kmem);
  X.nchunk = (M + kmax - 1) / kmax;
  X.K = ((M + X.nchunk - 1) / X.nchunk + 127) / 128 * 128;
  X.plane_bytes = (size_t)X.np * rows * X.K;
  const int32_t nstage = (int32_t)(X.K / 64);
  const int64_t one = (int64_t)p1 * kXT * kXT * 4;  // bytes of a pair's sums, per split
  // the blocks run one per CU
  const int64_t slots = std::max(num_cu, 1);
  X.nsplit = 1;
  X.per = nstage;
  double best = 0.0;
  for (int32_t s = 1; s <= std::min(nstage, 64); ++s) {
    if (s > 1 && s * X.npair * one > kXPartBytes) break;
    const int32_t pe = ((nstage + s - 1) / s + 1) & ~1, ns = (nstage + pe - 1) / pe;
    if (ns != s) continue;
    const double rounds = (double)(((int64_t)X.npair * p1 * ns + slots - 1) / slots);
    const double cost = rounds * ((double)pe + 12.0) + 0.5 * (double)X.npair * p1 * ns / slots;
    if (s == 1 || cost < best) {
      best = cost;
      X.nsplit = ns;
      X.per = pe;
    }
  }
  X.band = (int32_t)std::min<int64_t>(X.npair, kXPartBytes / (X.nsplit * one));
  X.part_bytes = (size_t)(X.nsplit * X.band * one);
  // about eight blocks a CU over the sample tiles
  const int32_t steps = (int32_t)((X.K + kResSnps - 1) / kResSnps);
  X.rsplit = std::min<int32_t>(steps, std::max<int32_t>(1, (int32_t)(8 * slots / nst)));
  X.rstep = (steps + X.rsplit - 1) / X.rsplit;
  X.rsplit = (steps + X.rstep - 1) / X.rstep;
  // left-out parts [K][4], their splits' and the chunk's sums, the digit tables
  X.tab_bytes = 64 * (size_t)X.K + 16 * (size_t)(X.rsplit + 1) * nst * 128 + 4 * (size_t)X.np * X.K;
  return X;
}
