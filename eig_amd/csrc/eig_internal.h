// Internal definitions shared by the HIP translation units of libeig_amd.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "../../include/eig_abi.h"
#include "plans.h"

// Sample tile of the selected-genotype layout: 128 samples = 8 x 32-bit words of
// 2-bit codes (sample 16w+i of the tile at bits 2i..2i+1 of word w).
constexpr int kTileS = 128;
constexpr int kTileWords = kTileS / 16;

// Largest K of loadings/lsqproject; the fxscal buffer holds K scales in its first
// kMaxK slots and xmean = mean*fancy after them.
constexpr int kMaxK = 16;

struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
};

struct eig_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr;  // begin of the stage under way
  std::string err;
  std::map<std::string, double> ms;
  // stage times: the events around each stage's last run, read when they are asked for
  struct Stage {
    hipEvent_t begin = nullptr, end = nullptr;
  };
  std::map<std::string, Stage> stages;
  int num_cu = 0;

  // genotypes as loaded (GENO row layout)
  DevBuf geno;
  int64_t rlen = 0, nsnp = 0;
  int32_t nind = 0;

  // selection of axis samples and its tile layout sel[(st*nsnp + m)*8 + w]
  DevBuf xindex, sel;
  int32_t nrows = 0, nst = 0;
  bool have_sel = false;
  bool sel_all = false;  // every loaded individual, in order
  // the same codes regrouped per 64-SNP group for the split-BF16 XTX (built on
  // first use after each selection)
  DevBuf selg;
  bool have_selg = false;
  // the split-BF16 SYRK's operand codes: per 64-SNP group, sample and k-slot half,
  // 16 bytes, each the LDS byte offset of a table entry (built on first use)
  DevBuf selb;
  bool have_selb = false;

  // per-SNP statistics (device)
  DevBuf c0, c1, nmiss, status, mean, fancy;
  DevBuf lev;    // double [nsnp][4] : levels of g = 0,1,2 and 0 for missing
  DevBuf levbf;  // uint32 [nsnp][4] : bf16 hi (low half) | bf16 lo (high half)
  DevBuf live;   // uint8 [nsnp]
  bool have_live = false;          // live mask of the last eig_snpstats
  int32_t altnorm = 1, fancynorm = 1;  // normalisation of the last eig_snpstats
  bool have_stats = false;
  // lsqproject fill table of usepopsformissing: [nsnp][npop] doubles, then nind types
  DevBuf fill;

  // XTX (normalised, row-major nrows x nrows) and partial sums
  DevBuf xtx, part;
  // FP64 form on the integer matrix cores: digit planes, tables, INT32 sums, pair list
  DevBuf xdplanes, xdtab, xdpart, xdmisc;
  bool have_xtx = false;
  // in use: XTX's workspaces, the eigensolver's, the regrouped codes (eig_malloc)
  bool in_syrk = false, in_eigh = false, in_selg = false;

  // eigensolver
  DevBuf ework;
  DevBuf tribuf;     // the tridiagonalisation's exchange words
  DevBuf evecs_dev;  // nvec x nrows of the last eig_eigh_xtx
  DevBuf evall;      // all-vector eigensolves: every batch's tridiagonal-basis vectors
  int32_t last_nvec = 0;

  // loadings / projection
  DevBuf ffvecs, fxscal, projw, proj_out, use_dev, ignore_dev;
  int32_t last_K = 0;
  // device address of this GPU's static workspace of eig_lsqproject_noalloc (set by
  // eig_open through hipGetSymbolAddress; never the array's host-side name)
  void *noalloc = nullptr;
  size_t noalloc_bytes = 0;
  bool have_load = false;

  // generic scratch
  DevBuf scratch, scratch2, hostpin;
};

int eig_set_err(eig_ctx *ctx, int code, const char *fmt, ...);
int eig_ensure(eig_ctx *ctx, DevBuf &b, size_t bytes);
// device memory; where it does not fit, the workspaces that no call under way uses go first
hipError_t eig_malloc(eig_ctx *ctx, void **p, size_t bytes);
struct EigInUse {  // marks an entry point's workspaces in use while it lives
  explicit EigInUse(bool &f) : flag(f) { flag = true; }
  ~EigInUse() { flag = false; }
  bool &flag;
};
// Results to the caller's (pageable) memory.  The runtime's own copies wait for each one,
// and move 12 GB/s.  get() queues a small copy into pinned memory, and the caller's memory
// is filled in wait(); a large one is done at once by several threads, each with two pinned
// pieces, one arriving while the other is copied on.  One at a time per context.
class EigFetch {
 public:
  explicit EigFetch(eig_ctx *ctx) : ctx_(ctx) {}
  int get(void *dst, const void *src, size_t bytes);
  int wait();  // the stream is idle and everything is in place

 private:
  struct Piece {
    void *dst;
    size_t at, bytes;
  };
  int big(char *dst, const char *src, size_t bytes);
  eig_ctx *ctx_;
  std::vector<Piece> small_;
  size_t used_ = 0;
};
// a stage's events; its time is read by eig_last_ms, and nothing waits here
void eig_time_begin(eig_ctx *ctx);
void eig_time_end(eig_ctx *ctx, const char *what);

#define EIG_HIP(ctx, call)                                                        \
  do {                                                                            \
    hipError_t e_ = (call);                                                       \
    if (e_ != hipSuccess)                                                         \
      return eig_set_err((ctx), EIG_E_HIP, "%s:%d %s: %s", __FILE__, __LINE__,    \
                         #call, hipGetErrorString(e_));                           \
  } while (0)

#define EIG_TRY(expr)           \
  do {                          \
    int r_ = (expr);            \
    if (r_ != EIG_OK) return r_; \
  } while (0)

// ---- device helpers ---------------------------------------------------------
__device__ __host__ inline uint16_t eig_bf16_rne(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf/nan
  uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(r >> 16);
}

__device__ __host__ inline float eig_bf16_to_f32(uint16_t h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  __builtin_memcpy(&f, &u, 4);
  return f;
}

// internal launchers implemented in the kernel translation units
int eig_syrk_digits(eig_ctx *ctx, double *dst, int *done);
int eig_run_syrk(eig_ctx *ctx, int form, int bf16_block, double *trace_scale);
// builds ctx->selg: per sample tile st, 64-SNP group g and sample i, 16 bytes at
// [(st * ceil(M/64) + g) * 128 + i]; word 2h + (s >> 1), bits 16 (s & 1) + 2 j hold the
// code of SNP 16 s + k of the group, h = (k >> 2) & 1, j = (k & 3) | ((k >> 3) << 2)
constexpr int kGrp = 64;  // SNPs per group of the grouped code layout
int eig_ensure_selg(eig_ctx *ctx);
int eig_regroup(eig_ctx *ctx, int64_t g0, int64_t ng);  // a range of the groups, at ctx->selg
// internal: a helper's own small problem -- the context's published eigenvectors
// (used by the loadings) and its stage times are left untouched
int eig_run_eigh(eig_ctx *ctx, const double *d_a, int32_t n, int32_t nvec, double *evals,
                 double *evecs,
                 bool internal = false);

// Column-major FP64 GEMM on MFMA with dgemm's conventions, batched by strides:
// C_b = alpha op(A_b) op(B_b) + beta C_b (C is not read when beta == 0).  lower: only
// the 64 x 64 tiles on or below the diagonal are formed (m == n).  Launched on `st`.
int eig_gemm_f64(eig_ctx *ctx, hipStream_t st, bool ta, bool tb, int64_t m, int64_t n, int64_t k,
                 double alpha, const double *A, int64_t lda, int64_t sA, const double *B,
                 int64_t ldb, int64_t sB, double beta, double *C, int64_t ldc, int64_t sC,
                 int32_t batch, bool lower = false);
// the same product with k cut into parts where its tiles are few; part: room for the parts'
// m x n results (part_doubles of them; parts that do not fit are not made)
int eig_gemm_f64_long(eig_ctx *ctx, hipStream_t st, bool ta, bool tb, int64_t m, int64_t n, int64_t k,
                      double alpha, const double *A, int64_t lda, const double *B, int64_t ldb,
                      double beta, double *C, int64_t ldc, bool lower, double *part,
                      size_t part_doubles);

// lsqproject's population fill table (usepopsformissing) from the loaded genotypes and
// the current ignore mask: types itype[q] (nind host entries, < 0 = none), npop types,
// use[q] the individuals projected, K the axes.  *fill = device table [nsnp][npop] (NaN:
// no data), *d_itype = the types on the device.
int eig_lsq_filltab(eig_ctx *ctx, const int32_t *use, const int32_t *itype, int32_t npop,
                    int32_t K, double **fill, const int32_t **d_itype);

// ---- products of packed codes with FP64 columns (codes.hip) ------------------
// The code words of a set of rows: row r's words pairs q = 0..3 of stage b (128 codes)
// at row base + b * KB + (q >> 1) * QH + (q & 1) * 8; row base = rows[r], or base +
// (r >> 7) * RT + (r & 127) * RS.  nword 16-code words per row are valid.
enum { kCodeLinear = 0, kCodeGrouped = 1, kCodeBytes = 2 };
struct CodeView {
  const uint8_t *base;
  const uint8_t *const *rows;
  int64_t RT, RS, KB, QH;
  int64_t nrow, nword;
  int32_t layout;
};
// columns: what kind of values, and where they are (see col_value)
enum { kColPanel, kColAxes, kColLevB, kColFx, kColLsqR, kColLsqG };
struct CodeCols {
  int kind;
  const double *a;
  int64_t ld, n;
  const double *lev = nullptr, *fancy = nullptr, *xmean = nullptr;
  const uint8_t *ignore = nullptr;
  const double *fxscal = nullptr;
  int32_t K = 0;
};
int eig_codes_scales(eig_ctx *ctx, const CodesPlan &P, const CodeCols &cols, void *head, hipStream_t st);
int eig_codes_restart(eig_ctx *ctx, const CodesPlan &P, void *head, hipStream_t st);
int eig_codes_build(eig_ctx *ctx, const CodesPlan &P, const CodeCols &cols, int32_t layout, int64_t b0,
                    void *head, void *dig, hipStream_t st);
hipError_t eig_codes_product(const CodesPlan &P, const CodeView &v, const void *dig, void *part,
                             bool accum, hipStream_t st);
hipError_t eig_codes_sum(const CodesPlan &P, int64_t nrow, const void *head, const void *part, double scale,
                         double *out, int64_t ldr, int64_t ldc, int32_t Cpad, bool add, hipStream_t st);
struct CodeRows {
  const uint8_t *row[16];
  int32_t n;
};
size_t eig_codes_small_bytes(const CodesPlan &P);
hipError_t eig_codes_small(const CodesPlan &P, const CodeRows &rows, int64_t nword, const void *head,
                           const void *dig, void *part, double *out, int64_t ldr, hipStream_t st);
int eig_codes_mul(eig_ctx *ctx, const CodesPlan &P, const CodeView &v, const CodeCols &cols, int64_t b0,
                  void *head, void *dig, void *part, bool accum, hipStream_t st);
int eig_codes_out_sum(eig_ctx *ctx, const CodesPlan &P, int64_t nrow, const void *head, const void *part,
                      double scale, double *out, int64_t ldr, int64_t ldc, int32_t Cpad, bool add,
                      hipStream_t st);
int eig_codes_samples(eig_ctx *ctx, const CodesPlan &P, const CodeCols &cols, char *ws, int64_t nrow,
                      double scale, double *out, int64_t ldr, int64_t ldc, int32_t Cpad, hipStream_t st);
int eig_codes_out_pair(eig_ctx *ctx, const CodesPlan &P, int64_t nrow, const void *head, const void *part,
                       const double *lev, const uint8_t *ignore, double scale, double *out, int64_t ldr,
                       int64_t ldc, hipStream_t st);
