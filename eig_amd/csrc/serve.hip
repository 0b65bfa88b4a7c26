// lsqproject serving: a request loop over a device-resident reference panel.
//
// The panel is the digit operands (codes.hip) of the projection rows e_m = fxscal .*
// ffvecs[:,m] times the fancy scale and xmean = mean*fancy, for the right-hand sides, and
// of the products e_m e_m^T, for the normal matrices, built once on the device from a
// context whose loadings are current.  Requests of 1..max_batch query samples arrive as
// sample-major packed rows (SNP m of a sample at byte m/4, bits 7-6, 5-4, 3-2, 1-0 for
// m%4 = 0..3, code 3 = missing).  A worker thread admits pending requests into free lanes:
// each lane is a stream with its own descriptor, row, partial-sum and output memory.
// Requests that arrive while other lanes are on the device are batched into the next free
// lane, so their work overlaps.
//
// Per sample the arithmetic is lsqproj + regressit + solvit (smartpca.c:4606-4757,
// regsubs.c:8-74, linsubs.c:296-393): over the sample's observed, kept SNPs the
// Gram co = sum e_m e_m^T and rhs rr = sum e_m x_m with x = g*fancy - xmean
// (fixxrow, qpsubs.c:338-349), then Cholesky (choldc/cholsl order).  The sums are exact
// integers on the panel's grid, whatever kernel and splits a batch takes, so a sample's
// result depends on its own row only, never on the other samples of its batch.
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <memory>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <vector>

#include "eig_internal.h"

constexpr int kSrvMaxK = 16;
constexpr int kSrvMaxBatch = 1024;  // samples per lane (descriptor capacity)
constexpr int kSrvMaxLanes = 8;

struct SrvDesc {
  const uint8_t *rows[kSrvMaxBatch];
};

// ------------------------------------------------------------------ kernels
// Cholesky solve per sample (choldc + cholsl order) on the packed triangle.
// out[q * (K + 2) + j]: coefficients, then status (0 solved, 1 <= K observed,
// 2 Cholesky failed or NaN), then the observed-SNP count.
template <int K>
// sums: per sample the triangle, the right-hand side and the observed count.  out is host
// memory: the few results leave with the kernel, without a copy of their own behind it.
__global__ __launch_bounds__(64) void k_srv_solve(int32_t n, const double *__restrict__ sums,
                                                  double *__restrict__ out) {
  constexpr int nP = K * (K + 1) / 2, W = nP + K + 1;
  for (int32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
    double A[nP], b[K], p[K], x[K];
#pragma unroll
    for (int i = 0; i < nP; ++i) A[i] = sums[(int64_t)q * W + i];
#pragma unroll
    for (int i = 0; i < K; ++i) b[i] = sums[(int64_t)q * W + nP + i];
    const double kk = sums[(int64_t)q * W + nP + K];
    double *o = out + (int64_t)q * (K + 2);
    o[K + 1] = kk;
    if (kk <= (double)K) {
#pragma unroll
      for (int j = 0; j < K; ++j) o[j] = 0.0;
      o[K] = 1.0;
      continue;
    }
    bool bad = false;
#pragma unroll
    for (int i = 0; i < nP; ++i) bad |= isnan(A[i]);
#pragma unroll
    for (int i = 0; i < K; ++i) bad |= isnan(b[i]);
    // P(i, j), i <= j, holds the input a[i][j] until step (i, j) overwrites it with L[j][i]
#define SRV_P(i, j) A[(i) * K - (i) * ((i) - 1) / 2 + ((j) - (i))]
#pragma unroll
    for (int i = 0; i < K; ++i) {
#pragma unroll
      for (int j = i; j < K; ++j) {
        double s = SRV_P(i, j);
#pragma unroll
        for (int k = i - 1; k >= 0; --k) s -= SRV_P(k, i) * SRV_P(k, j);
        if (i == j) {
          bad |= !(s > 0.0);
          p[i] = sqrt(s > 0.0 ? s : 1.0);
        } else {
          SRV_P(i, j) = s / p[i];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
      double s = b[i];
#pragma unroll
      for (int k = i - 1; k >= 0; --k) s -= SRV_P(k, i) * x[k];
      x[i] = s / p[i];
    }
#pragma unroll
    for (int i = K - 1; i >= 0; --i) {
      double s = x[i];
#pragma unroll
      for (int k = i + 1; k < K; ++k) s -= SRV_P(i, k) * x[k];
      x[i] = s / p[i];
    }
#undef SRV_P
#pragma unroll
    for (int j = 0; j < K; ++j) o[j] = bad ? 0.0 : x[j];
    o[K] = bad ? 2.0 : 0.0;
  }
}

// ------------------------------------------------------------------ host side
using Clock = std::chrono::steady_clock;

struct SrvReq {
  int64_t id = 0;
  int32_t nq = 0;
  const uint8_t *rows = nullptr;
  int64_t stride = 0;
  bool on_device = false;
  Clock::time_point t_submit, t_done;
  bool done = false;
  int err = EIG_OK;
  std::vector<double> coords;  // nq x K
  std::vector<int32_t> status;
};

struct SrvLane {
  hipStream_t stream = nullptr;
  hipEvent_t done = nullptr;
  SrvDesc *desc_h = nullptr, *desc_d = nullptr;
  uint8_t *rows_d = nullptr;
  char *partial_d = nullptr;
  double *sums_d = nullptr, *out_h = nullptr;
  std::vector<std::shared_ptr<SrvReq>> reqs;
  std::vector<int32_t> offs;
  bool busy = false;
};

struct eig_server {
  int device = 0;
  int32_t K = 0, nP = 0, W = 0;
  int64_t M = 0, rowbytes = 0, rowpad = 0;
  int32_t nlanes = 0, max_batch = 0;
  int32_t chunk = 0, smax = 1;
  int num_cu = 0;
  double eigscale[kSrvMaxK];
  // the panel: scales and digit operands of the right-hand sides and of the normal matrices
  CodesPlan pr, pg;
  char *panel_d = nullptr;
  void *head_r = nullptr, *head_g = nullptr, *dig_r = nullptr, *dig_g = nullptr;
  size_t part_bytes = 0;  // of a lane
  SrvLane lane[kSrvMaxLanes];

  std::mutex mu;
  std::condition_variable cv_work, cv_done;
  std::deque<std::shared_ptr<SrvReq>> pending;
  std::unordered_map<int64_t, std::shared_ptr<SrvReq>> reqs;
  int64_t next_id = 1;
  bool stopping = false;
  std::thread worker;
  std::string err;
  int64_t nbatches = 0, nsamples = 0;
};

static int srv_err(eig_server *s, int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  if (s) s->err = buf;
  return code;
}

#define SRV_HIP(s, call)                                                                      \
  do {                                                                                        \
    hipError_t e_ = (call);                                                                   \
    if (e_ != hipSuccess)                                                                     \
      return srv_err((s), EIG_E_HIP, "%s:%d %s: %s", __FILE__, __LINE__, #call,               \
                     hipGetErrorString(e_));                                                  \
  } while (0)

// a batch's plan: splits of at least `chunk` SNPs, as many as help and 32 MiB of sums hold
static CodesPlan srv_plan(const eig_server *s, int mode, int32_t n) {
  const int32_t C = mode == kCdSum ? s->K + 1 : s->nP;
  const int64_t nblk = (s->M + 127) / 128;
  const CodesPlan one = eig_codes_plan(s->num_cu, mode, C, n, nblk, 1);
  const size_t per = one.part_bytes / one.nsplit;
  return eig_codes_plan(s->num_cu, mode, C, n, nblk,
                        (int32_t)std::min<int64_t>(s->smax, std::max<int64_t>(1, ((int64_t)32 << 20) / (int64_t)per)));
}

#define SRV_KCASE(n, ...) \
  case n: {               \
    constexpr int KC = n; \
    __VA_ARGS__;          \
  } break;
#define SRV_KSWITCH(s, k, ...)                                                              \
  switch (k) {                                                                              \
    SRV_KCASE(1, __VA_ARGS__) SRV_KCASE(2, __VA_ARGS__) SRV_KCASE(3, __VA_ARGS__)            \
    SRV_KCASE(4, __VA_ARGS__) SRV_KCASE(5, __VA_ARGS__) SRV_KCASE(6, __VA_ARGS__)            \
    SRV_KCASE(7, __VA_ARGS__) SRV_KCASE(8, __VA_ARGS__) SRV_KCASE(9, __VA_ARGS__)            \
    SRV_KCASE(10, __VA_ARGS__) SRV_KCASE(11, __VA_ARGS__) SRV_KCASE(12, __VA_ARGS__)         \
    SRV_KCASE(13, __VA_ARGS__) SRV_KCASE(14, __VA_ARGS__) SRV_KCASE(15, __VA_ARGS__)         \
    SRV_KCASE(16, __VA_ARGS__)                                                              \
    default:                                                                                \
      return srv_err(s, EIG_E_ARG, "K out of range");                                       \
  }

// A batch's normal equations and solutions on its lane's stream.  Up to 16 samples fill one
// row tile: the digits, 355 MB at 600,000 SNPs and K = 10, stream through once
// (k_cd_stream: 76 us, and 0.11 ms from submit to result, where FP64 sums of a lane per
// sample took 0.82).  More share each digit operand through LDS (k_cd_mul: 112 samples in
// 0.19 ms, 586 in 0.49).
static int srv_launch(eig_server *s, SrvLane &L, int32_t n) {
  hipStream_t st = L.stream;
  const int64_t nword = s->rowpad / 4;
  if (n <= 16) {
    CodeRows rows;
    rows.n = n;
    for (int32_t i = 0; i < 16; ++i) rows.row[i] = L.desc_h->rows[i < n ? i : 0];
    char *sg = L.partial_d + eig_codes_small_bytes(s->pr);
    SRV_HIP(s, eig_codes_small(s->pg, rows, nword, s->head_g, s->dig_g, sg, L.sums_d, s->W, st));
    SRV_HIP(s, eig_codes_small(s->pr, rows, nword, s->head_r, s->dig_r, L.partial_d, L.sums_d + s->nP,
                               s->W, st));
  } else {
    SRV_HIP(s, hipMemcpyAsync(L.desc_d, L.desc_h, sizeof(void *) * (size_t)n, hipMemcpyHostToDevice, st));
    const CodeView v{nullptr, L.desc_d->rows, 0, 0, 32, 16, n, nword, kCodeBytes};
    const CodesPlan pr = srv_plan(s, kCdSum, n), pg = srv_plan(s, kCdMiss, n);
    char *sg = L.partial_d + (pr.part_bytes + 255) / 256 * 256;
    SRV_HIP(s, eig_codes_product(pg, v, s->dig_g, sg, false, st));
    SRV_HIP(s, eig_codes_product(pr, v, s->dig_r, L.partial_d, false, st));
    SRV_HIP(s, eig_codes_sum(pg, n, s->head_g, sg, 1.0, L.sums_d, s->W, 1, s->nP, false, st));
    SRV_HIP(s, eig_codes_sum(pr, n, s->head_r, L.partial_d, 1.0, L.sums_d + s->nP, s->W, 1, s->K + 1,
                             false, st));
  }
  SRV_KSWITCH(s, s->K,
              hipLaunchKernelGGL((k_srv_solve<KC>), dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, n,
                                 (const double *)L.sums_d, L.out_h));
  SRV_HIP(s, hipGetLastError());
  return EIG_OK;
}

// Launch one batch on a lane (worker thread, no lock held).
static int srv_dispatch(eig_server *s, SrvLane &L) {
  hipStream_t st = L.stream;
  int32_t off = 0;
  L.offs.clear();
  for (auto &r : L.reqs) {
    L.offs.push_back(off);
    if (r->on_device) {
      for (int32_t i = 0; i < r->nq; ++i) L.desc_h->rows[off + i] = r->rows + (int64_t)i * r->stride;
    } else {
      uint8_t *dst = L.rows_d + (int64_t)off * s->rowpad;
      SRV_HIP(s, hipMemcpy2DAsync(dst, (size_t)s->rowpad, r->rows, (size_t)r->stride,
                                  (size_t)s->rowbytes, (size_t)r->nq, hipMemcpyHostToDevice, st));
      for (int32_t i = 0; i < r->nq; ++i) L.desc_h->rows[off + i] = dst + (int64_t)i * s->rowpad;
    }
    off += r->nq;
  }
  int rc = srv_launch(s, L, off);
  if (rc != EIG_OK) return rc;
  SRV_HIP(s, hipEventRecord(L.done, st));
  return EIG_OK;
}

// Results of a finished lane (worker thread, lock held).  Within a request, a
// failed Cholesky keeps the previous sample's answer (regsubs.c:51-53, regans
// zeroed per call at smartpca.c:4656); coordinates are eigscale * a
// (smartpca.c:1556-1564).
static void srv_finish(eig_server *s, SrvLane &L, int err) {
  const int K = s->K;
  const auto now = Clock::now();
  for (size_t r = 0; r < L.reqs.size(); ++r) {
    SrvReq &q = *L.reqs[r];
    q.err = err;
    q.coords.assign((size_t)q.nq * K, 0.0);
    q.status.assign((size_t)q.nq, 0);
    double last[kSrvMaxK] = {0.0};
    for (int32_t i = 0; i < q.nq && err == EIG_OK; ++i) {
      const double *o = L.out_h + (size_t)(L.offs[r] + i) * (K + 2);
      const int stt = (int)o[K];
      q.status[i] = stt;
      if (stt == 0)
        for (int j = 0; j < K; ++j) last[j] = o[j];
      if (stt != 1)
        for (int j = 0; j < K; ++j) q.coords[(size_t)i * K + j] = s->eigscale[j] * last[j];
    }
    q.t_done = now;
    q.done = true;
  }
  s->nbatches += 1;
  L.reqs.clear();
  L.busy = false;
}

// The worker looks for finished batches without a pause for this long after it last started or
// finished one: a batch takes 0.1 to a few tenths of a millisecond, and a timed wait of 20 us
// returns after 70 to 80.  Longer ones (large batches, host rows, a card that others use) are
// waited for with such waits, not with the core.
constexpr auto kSrvSpin = std::chrono::milliseconds(1);

static void srv_worker(eig_server *s) {
  hipSetDevice(s->device);
  std::unique_lock<std::mutex> lk(s->mu);
  auto spin_end = Clock::now();
  for (;;) {
    bool progressed = false;
    // completions; the lanes are this thread's alone, so it asks without the lock that submit
    // and poll need
    hipError_t state[kSrvMaxLanes];
    lk.unlock();
    for (int l = 0; l < s->nlanes; ++l)
      state[l] = s->lane[l].busy ? hipEventQuery(s->lane[l].done) : hipErrorNotReady;
    lk.lock();
    for (int l = 0; l < s->nlanes; ++l) {
      SrvLane &L = s->lane[l];
      const hipError_t q = state[l];
      if (!L.busy || q == hipErrorNotReady) continue;
      srv_finish(s, L, q == hipSuccess ? EIG_OK : EIG_E_HIP);
      if (q != hipSuccess) s->err = hipGetErrorString(q);
      progressed = true;
    }
    if (progressed) s->cv_done.notify_all();
    // admissions: FIFO requests into free lanes, as many as a lane holds
    for (int l = 0; l < s->nlanes && !s->pending.empty(); ++l) {
      SrvLane &L = s->lane[l];
      if (L.busy) continue;
      int32_t tot = 0;
      while (!s->pending.empty() && tot + s->pending.front()->nq <= s->max_batch) {
        tot += s->pending.front()->nq;
        L.reqs.push_back(s->pending.front());
        s->pending.pop_front();
      }
      L.busy = true;
      s->nsamples += tot;
      lk.unlock();
      int rc = srv_dispatch(s, L);
      lk.lock();
      if (rc != EIG_OK) {
        srv_finish(s, L, rc);
        s->cv_done.notify_all();
      }
      progressed = true;
    }
    bool any_busy = false;
    for (int l = 0; l < s->nlanes; ++l) any_busy |= s->lane[l].busy;
    if (s->stopping && !any_busy && s->pending.empty()) break;
    if (progressed) {
      spin_end = Clock::now() + kSrvSpin;
      continue;
    }
    if (!any_busy) {
      s->cv_work.wait(lk, [s] { return s->stopping || !s->pending.empty(); });
    } else if (Clock::now() < spin_end) {
      lk.unlock();
      std::this_thread::yield();
      lk.lock();
    } else {
      s->cv_work.wait_for(lk, std::chrono::microseconds(20));
    }
  }
}

static void srv_free(eig_server *s) {
  for (int l = 0; l < kSrvMaxLanes; ++l) {
    SrvLane &L = s->lane[l];
    if (L.done) hipEventDestroy(L.done);
    if (L.stream) hipStreamDestroy(L.stream);
    if (L.desc_h) hipHostFree(L.desc_h);
    if (L.out_h) hipHostFree(L.out_h);
    if (L.desc_d) hipFree(L.desc_d);
    if (L.rows_d) hipFree(L.rows_d);
    if (L.partial_d) hipFree(L.partial_d);
    if (L.sums_d) hipFree(L.sums_d);
  }
  if (s->panel_d) hipFree(s->panel_d);
  delete s;
}

static int srv_alloc_lane(eig_ctx *ctx, eig_server *s, SrvLane &L) {
  SRV_HIP(s, hipStreamCreateWithFlags(&L.stream, hipStreamNonBlocking));
  SRV_HIP(s, hipEventCreateWithFlags(&L.done, hipEventDisableTiming));
  SRV_HIP(s, hipHostMalloc((void **)&L.desc_h, sizeof(SrvDesc), hipHostMallocDefault));
  SRV_HIP(s, hipHostMalloc((void **)&L.out_h, sizeof(double) * s->max_batch * (s->K + 2),
                           hipHostMallocDefault));
  SRV_HIP(s, eig_malloc(ctx, (void **)&L.desc_d, sizeof(SrvDesc)));
  SRV_HIP(s, eig_malloc(ctx, (void **)&L.rows_d, (size_t)s->max_batch * s->rowpad));
  SRV_HIP(s, eig_malloc(ctx, (void **)&L.partial_d, s->part_bytes));
  SRV_HIP(s, eig_malloc(ctx, (void **)&L.sums_d, sizeof(double) * s->W * s->max_batch));
  std::memset(L.desc_h, 0, sizeof(SrvDesc));
  return EIG_OK;
}

extern "C" int eig_server_start(eig_ctx *ctx, const double *eigscale, int32_t nlanes,
                                int32_t max_batch, int32_t chunk, eig_server **out) {
  if (!ctx || !out) return eig_set_err(ctx, EIG_E_ARG, "eig_server_start: null argument");
  *out = nullptr;
  if (!ctx->have_load)
    return eig_set_err(ctx, EIG_E_STATE, "eig_server_start before eig_loadings");
  if (nlanes <= 0) nlanes = 4;
  if (max_batch <= 0) max_batch = kSrvMaxBatch;
  if (nlanes > kSrvMaxLanes || max_batch > kSrvMaxBatch)
    return eig_set_err(ctx, EIG_E_ARG, "eig_server_start: nlanes <= %d, max_batch <= %d",
                       kSrvMaxLanes, kSrvMaxBatch);
  if (chunk < 0 || chunk % 64 != 0)
    return eig_set_err(ctx, EIG_E_ARG, "eig_server_start: chunk must be a multiple of 64");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  EIG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  eig_server *s = new eig_server();
  s->device = ctx->device;
  s->num_cu = ctx->num_cu;
  s->K = ctx->last_K;
  s->nP = s->K * (s->K + 1) / 2;
  s->W = s->nP + s->K + 1;
  s->M = ctx->nsnp;
  s->rowbytes = (s->M + 3) / 4;
  s->rowpad = ((s->M + 63) / 64) * 16;
  s->nlanes = nlanes;
  s->max_batch = max_batch;
  for (int j = 0; j < kSrvMaxK; ++j) s->eigscale[j] = (eigscale && j < s->K) ? eigscale[j] : 1.0;
  // splits of a batch: at least `chunk` SNPs each; 4,096 when the caller leaves it (at
  // 600,000 SNPs, K = 10, 112 samples alone and a burst of 963 in 24 requests take 0.17 and
  // 0.85 ms with 1,024, 0.19 and 0.74 with 4,096, 0.45 and 0.85 with 16,384)
  s->chunk = chunk > 0 ? chunk : 4096;
  s->smax = (int32_t)std::min<int64_t>(512, std::max<int64_t>(1, s->M / std::max(s->chunk, 128)));
  auto fail = [&](int rc) {
    ctx->err = s->err;
    srv_free(s);
    return rc;
  };
  {
    const double *fx = (const double *)ctx->fxscal.p;
    CodeCols cr{kColLsqR, (const double *)ctx->ffvecs.p, s->M, s->M};
    cr.fancy = (const double *)ctx->fancy.p;
    cr.xmean = fx + kMaxK;
    cr.ignore = (const uint8_t *)ctx->ignore_dev.p;
    cr.fxscal = fx;
    cr.K = s->K;
    CodeCols cg = cr;
    cg.kind = kColLsqG;
    s->pr = srv_plan(s, kCdSum, 16);
    s->pg = srv_plan(s, kCdMiss, 16);
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    if (eig_malloc(ctx, (void **)&s->panel_d, s->pr.head_bytes + s->pg.head_bytes + up(s->pr.dig_bytes) +
                                                  s->pg.dig_bytes) != hipSuccess)
      return fail(srv_err(s, EIG_E_NOMEM, "panel allocation"));
    s->head_r = s->panel_d;
    s->head_g = s->panel_d + s->pr.head_bytes;
    s->dig_r = (char *)s->head_g + s->pg.head_bytes;
    s->dig_g = (char *)s->dig_r + up(s->pr.dig_bytes);
    for (int g = 0; g < 2; ++g) {
      const CodesPlan &P = g ? s->pg : s->pr;
      const CodeCols &c = g ? cg : cr;
      void *head = g ? s->head_g : s->head_r, *dig = g ? s->dig_g : s->dig_r;
      int rc = eig_codes_scales(ctx, P, c, head, ctx->stream);
      if (rc == EIG_OK) rc = eig_codes_build(ctx, P, c, kCodeBytes, 0, head, dig, ctx->stream);
      if (rc != EIG_OK) return fail(srv_err(s, rc, "panel build failed"));
    }
    if (hipStreamSynchronize(ctx->stream) != hipSuccess)
      return fail(srv_err(s, EIG_E_HIP, "panel build failed"));
    // a lane's partial sums: the small product's, or any batch's
    s->part_bytes = eig_codes_small_bytes(s->pr) + eig_codes_small_bytes(s->pg);
    for (int32_t n = 17; n <= max_batch; ++n)
      s->part_bytes = std::max(s->part_bytes, up(srv_plan(s, kCdSum, n).part_bytes) +
                                                  up(srv_plan(s, kCdMiss, n).part_bytes));
  }
  for (int l = 0; l < nlanes; ++l) {
    SrvLane &L = s->lane[l];
    int rc = srv_alloc_lane(ctx, s, L);
    if (rc != EIG_OK) return fail(rc);
    // a batch of each kind on the lane, so that the first request does not pay for the
    // stream's queue and the first touch of its memory (any byte is a valid row)
    const int32_t nw = std::min(32, max_batch);
    if (hipMemsetAsync(L.rows_d, 0, (size_t)nw * s->rowpad, L.stream) != hipSuccess)
      return fail(srv_err(s, EIG_E_HIP, "lane start"));
    for (int32_t i = 0; i < nw; ++i) L.desc_h->rows[i] = L.rows_d + (int64_t)i * s->rowpad;
    for (int32_t n : {1, nw}) {
      rc = srv_launch(s, L, n);
      if (rc != EIG_OK) return fail(rc);
    }
    if (hipEventRecord(L.done, L.stream) != hipSuccess || hipStreamSynchronize(L.stream) != hipSuccess)
      return fail(srv_err(s, EIG_E_HIP, "lane start"));
  }
  s->worker = std::thread(srv_worker, s);
  *out = s;
  return EIG_OK;
}

extern "C" int eig_server_submit(eig_server *s, const uint8_t *rows, int64_t stride, int32_t nq,
                                 int32_t on_device, int64_t *ticket) {
  if (!s || !rows || !ticket) return srv_err(s, EIG_E_ARG, "eig_server_submit: null argument");
  if (nq < 1 || nq > s->max_batch)
    return srv_err(s, EIG_E_ARG, "eig_server_submit: nq must be in [1, %d]", s->max_batch);
  if (on_device) {
    if (stride < s->rowpad || stride % 16 != 0 || ((uintptr_t)rows & 15) != 0)
      return srv_err(s, EIG_E_ARG,
                     "eig_server_submit: device rows need 16-byte alignment and stride >= %lld",
                     (long long)s->rowpad);
  } else if (stride < s->rowbytes) {
    return srv_err(s, EIG_E_ARG, "eig_server_submit: stride < %lld", (long long)s->rowbytes);
  }
  auto r = std::make_shared<SrvReq>();
  r->nq = nq;
  r->rows = rows;
  r->stride = stride;
  r->on_device = on_device != 0;
  r->t_submit = Clock::now();
  {
    std::lock_guard<std::mutex> g(s->mu);
    if (s->stopping) return srv_err(s, EIG_E_STATE, "eig_server_submit after stop");
    r->id = s->next_id++;
    s->reqs[r->id] = r;
    s->pending.push_back(r);
  }
  s->cv_work.notify_one();
  *ticket = r->id;
  return EIG_OK;
}

extern "C" int eig_server_poll(eig_server *s, int64_t ticket, int32_t wait, double *coords,
                               int32_t *status, double *latency_ms) {
  if (!s) return EIG_E_ARG;
  std::unique_lock<std::mutex> lk(s->mu);
  auto it = s->reqs.find(ticket);
  if (it == s->reqs.end()) return srv_err(s, EIG_E_ARG, "eig_server_poll: unknown ticket");
  std::shared_ptr<SrvReq> r = it->second;
  if (!r->done) {
    if (!wait) return EIG_PENDING;
    s->cv_done.wait(lk, [&] { return r->done; });
  }
  s->reqs.erase(it);
  if (r->err != EIG_OK) return srv_err(s, r->err, "request failed: %s", s->err.c_str());
  if (coords) std::memcpy(coords, r->coords.data(), sizeof(double) * r->coords.size());
  if (status) std::memcpy(status, r->status.data(), sizeof(int32_t) * r->status.size());
  if (latency_ms)
    *latency_ms = std::chrono::duration<double, std::milli>(r->t_done - r->t_submit).count();
  return EIG_OK;
}

extern "C" int eig_server_info(eig_server *s, int32_t *K, int64_t *nsnp, int64_t *rowpad,
                               int32_t *chunk, int32_t *grid, int64_t *batches,
                               int64_t *samples) {
  if (!s) return EIG_E_ARG;
  std::lock_guard<std::mutex> g(s->mu);
  if (K) *K = s->K;
  if (nsnp) *nsnp = s->M;
  if (rowpad) *rowpad = s->rowpad;
  if (chunk) *chunk = s->chunk;
  if (grid) *grid = 2 * s->num_cu;
  if (batches) *batches = s->nbatches;
  if (samples) *samples = s->nsamples;
  return EIG_OK;
}

extern "C" const char *eig_server_error(const eig_server *s) {
  return s ? s->err.c_str() : "null server";
}

extern "C" void eig_server_stop(eig_server *s) {
  if (!s) return;
  {
    std::lock_guard<std::mutex> g(s->mu);
    s->stopping = true;
  }
  s->cv_work.notify_all();
  if (s->worker.joinable()) s->worker.join();
  hipSetDevice(s->device);
  for (int l = 0; l < s->nlanes; ++l)
    if (s->lane[l].stream) hipStreamSynchronize(s->lane[l].stream);
  srv_free(s);
}

// ------------------------------------------------------------------ synthetic queries
__device__ __host__ inline uint64_t srv_mix64(uint64_t x) {
  x ^= x >> 30;
  x *= 0xBF58476D1CE4E5B9ull;
  x ^= x >> 27;
  x *= 0x94D049BB133111EBull;
  x ^= x >> 31;
  return x;
}

// One thread per output byte: sample q, SNPs 4b..4b+3 (sample-major rows).
__global__ void k_synth_queries(uint8_t *__restrict__ rows, int64_t stride, int64_t nsnp,
                                int32_t nq, const uint32_t *__restrict__ thr,
                                const int32_t *__restrict__ pop,
                                const uint32_t *__restrict__ miss_thr, uint64_t seed) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= stride * nq) return;
  const int32_t q = (int32_t)(idx / stride);
  const int64_t b = idx - (int64_t)q * stride;
  uint32_t byte = 0;
  for (int k = 0; k < 4; ++k) {
    const int64_t m = 4 * b + k;
    uint32_t code = 3;
    if (m < nsnp) {
      const uint64_t key = (uint64_t)q * (uint64_t)nsnp + (uint64_t)m;
      const uint64_t h1 = srv_mix64(seed + (key + 1) * 0x9E3779B97F4A7C15ull);
      const uint64_t h2 = srv_mix64(h1 ^ 0x5851F42D4C957F2Dull);
      const uint32_t t = thr[(int64_t)pop[q] * nsnp + m];
      const uint32_t g = ((uint32_t)h1 < t ? 1u : 0u) + ((uint32_t)(h1 >> 32) < t ? 1u : 0u);
      code = ((uint32_t)h2 < miss_thr[q]) ? 3u : g;
    }
    byte |= code << (6 - 2 * k);
  }
  rows[idx] = (uint8_t)byte;
}

extern "C" int eig_synth_queries(eig_ctx *ctx, int64_t nsnp, int32_t nq, int32_t npop,
                                 const uint32_t *thr, const int32_t *pop,
                                 const uint32_t *miss_thr, uint64_t seed, uint8_t *rows_dev,
                                 int64_t stride) {
  if (!ctx || nsnp <= 0 || nq <= 0 || npop <= 0 || !thr || !pop || !miss_thr || !rows_dev ||
      stride < (nsnp + 3) / 4)
    return eig_set_err(ctx, EIG_E_ARG, "eig_synth_queries: bad args");
  for (int32_t q = 0; q < nq; ++q)
    if (pop[q] < 0 || pop[q] >= npop) return eig_set_err(ctx, EIG_E_ARG, "pop out of range");
  EIG_HIP(ctx, hipSetDevice(ctx->device));
  const size_t tb = sizeof(uint32_t) * (size_t)npop * nsnp;
  const size_t pb = ((sizeof(int32_t) * (size_t)nq + 255) / 256) * 256;
  EIG_TRY(eig_ensure(ctx, ctx->scratch, tb + 2 * pb));
  uint32_t *d_thr = (uint32_t *)ctx->scratch.p;
  int32_t *d_pop = (int32_t *)((char *)ctx->scratch.p + tb);
  uint32_t *d_miss = (uint32_t *)((char *)ctx->scratch.p + tb + pb);
  hipStream_t st = ctx->stream;
  EIG_HIP(ctx, hipMemcpyAsync(d_thr, thr, tb, hipMemcpyHostToDevice, st));
  EIG_HIP(ctx, hipMemcpyAsync(d_pop, pop, sizeof(int32_t) * nq, hipMemcpyHostToDevice, st));
  EIG_HIP(ctx, hipMemcpyAsync(d_miss, miss_thr, sizeof(uint32_t) * nq, hipMemcpyHostToDevice, st));
  const int64_t total = stride * nq;
  hipLaunchKernelGGL(k_synth_queries, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     rows_dev, stride, nsnp, nq, (const uint32_t *)d_thr, (const int32_t *)d_pop,
                     (const uint32_t *)d_miss, seed);
  EIG_HIP(ctx, hipGetLastError());
  EIG_HIP(ctx, hipStreamSynchronize(st));
  return EIG_OK;
}
