// bc.hip - boundary-condition time series applied on the device.
//
// One thread per element edge and river segment, which interpolates its series
// if it has one (IntrplForc, src/forcing.c:482-530; ApplyElemBc, :127-177;
// ApplyRiverBc, :214-244); where a great many have one, a launch of one thread
// per series interpolates them first.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/pihm_bc.h"
#include "common.hpp"
#include "ctx.hpp"
#include "tsinterp.hpp"

using namespace pihm;

namespace {

// One set of series: nrec records each, series-major.
struct BcSeries {
  int nrec;
  const double *ft, *v;
};

// code > 0: series code-1 (head); code < 0: series -code-1 (flux); 0: unchanged.
// Element edges first (edge-major, device order), then river segments.  The few
// entries that have a series interpolate it themselves, beside the many that
// only read their code: bound by the codes and one bisection's loads.
__global__ __launch_bounds__(kBlock) void k_bc(long n_edge, int nr, const int32_t *code_e, const int32_t *code_r,
                                               BcSeries se, BcSeries sr, double t, double *ebc, double *rbc) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_edge + nr) return;
  const bool edge = i < n_edge;
  const int c = edge ? code_e[i] : code_r[i - n_edge];
  if (c == 0) return;
  const BcSeries s = edge ? se : sr;
  const long k = (c > 0 ? c : -c) - 1;
  ts_interp<1>(s.ft + k * s.nrec, s.v + k * s.nrec, s.nrec, t, edge ? ebc + i : rbc + (i - n_edge), 1);
}

// Above kBcDirect entries with a series, in two launches: every series' value
// into a table, element series first, then the entries from the table (bound by
// the codes and the values written, whatever the length of the series).
__global__ __launch_bounds__(kBlock) void k_bc_interp(int nts_e, int nts_r, BcSeries se, BcSeries sr, double t,
                                                      double *val) {
  const int k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= nts_e + nts_r) return;
  const BcSeries s = k < nts_e ? se : sr;
  const long q = k < nts_e ? k : k - nts_e;
  ts_interp<1>(s.ft + q * s.nrec, s.v + q * s.nrec, s.nrec, t, val + k, 1);
}
__global__ __launch_bounds__(kBlock) void k_bc_scatter(long n_edge, int nr, const int32_t *code_e,
                                                       const int32_t *code_r, int nts_e, const double *val,
                                                       double *ebc, double *rbc) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n_edge + nr) return;
  const bool edge = i < n_edge;
  const int c = edge ? code_e[i] : code_r[i - n_edge];
  if (c == 0) return;
  const double v = val[(edge ? 0 : nts_e) + (c > 0 ? c : -c) - 1];
  if (edge) ebc[i] = v;
  else rbc[i - n_edge] = v;
}

// Entries with a series up to which they interpolate it themselves.  Measured
// (us per apply, one launch / two; series of 1,000 and of 20,000 records):
// the outer edges and the river segments of 200,000 triangles, 6,306 of 605,000
// entries, 4.7 / 5.8 and 6.1 / 6.8; a tenth of the edges drawn at random, 6,487
// of 60,533 entries 4.3 / 5.4 and 5.2 / 6.5, 19,462 of 181,500 5.0 / 5.7 and
// 6.8 / 6.5, 32,630 of 302,500 6.3 / 5.8 and 8.7 / 6.7, 65,114 of 605,000
// 10.9 / 6.6 and 15.6 / 7.5; all of 605,000 19.8 / 6.8 and 35.5 / 7.8.
constexpr long kBcDirect = 16384;

bool times_increase(const pihm_ts *s) {
  for (int k = 0; k < s->nts; k++)
    for (int r = 1; r < s->nrec; r++)
      if (!(s->ftime[(long)k * s->nrec + r] > s->ftime[(long)k * s->nrec + r - 1])) return false;
  return true;
}

}  // namespace

struct pihm_bc {
  pihm_ctx *ctx;
  int nts_e, nrec_e, nts_r, nrec_r;
  long n_edge;
  int nr;
  int32_t *code_e, *code_r;
  double *ft_e, *v_e, *ft_r, *v_r, *val;
  long ncoded;          // edges and segments with a series
  double t_lo, t_hi;    // the time range every series covers
  void *arena;
};

namespace pihm {
pihm_ctx *bc_context(const pihm_bc *b) { return b ? b->ctx : nullptr; }
}

extern "C" {

int pihm_bc_create(pihm_ctx *ctx, const int32_t *elem_type, const pihm_ts *ets, const int32_t *river_type,
                   const pihm_ts *rts, pihm_bc **out) {
  if (!out) return PIHM_ERR_ARG;
  *out = nullptr;
  if (!ctx || ctx->nmem != 1) return PIHM_ERR_ARG;
  const int ne = ctx->ne, nr = ctx->nr;
  const int nts_e = ets ? ets->nts : 0, nts_r = rts ? rts->nts : 0;
  for (const pihm_ts *s : {ets, rts})
    if (s && (s->nts < 0 || (s->nts > 0 && (s->nrec < 2 || !s->ftime || !s->value || !times_increase(s)))))
      return PIHM_ERR_ARG;
  std::vector<int32_t> ce(3L * ne, 0), cr(nr > 0 ? nr : 1, 0);
  if (elem_type)
    for (int p = 0; p < ne; p++)
      for (int j = 0; j < 3; j++) {
        const int c = elem_type[3L * ctx->perm[p] + j];
        if (c > nts_e || -c > nts_e) return PIHM_ERR_ARG;
        ce[(long)j * ne + p] = c;
      }
  if (river_type)
    for (int r = 0; r < nr; r++) {
      const long q = caller_river(ctx, r);
      const int c = q >= 0 ? river_type[q] : 0;
      if (c > nts_r || -c > nts_r) return PIHM_ERR_ARG;
      cr[r] = c;
    }
  pihm_bc *b = new pihm_bc();
  b->ctx = ctx;
  b->nts_e = nts_e;
  b->nrec_e = nts_e ? ets->nrec : 0;
  b->nts_r = nts_r;
  b->nrec_r = nts_r ? rts->nrec : 0;
  b->n_edge = 3L * ne;
  b->ncoded = 0;
  for (const int32_t c : ce) b->ncoded += c != 0;
  for (const int32_t c : cr) b->ncoded += c != 0;
  b->nr = nr;
  b->t_lo = -HUGE_VAL;
  b->t_hi = HUGE_VAL;
  for (const pihm_ts *s : {ets, rts})
    if (s)
      for (int k = 0; k < s->nts; k++) {
        b->t_lo = std::max(b->t_lo, s->ftime[(long)k * s->nrec]);
        b->t_hi = std::min(b->t_hi, s->ftime[(long)k * s->nrec + s->nrec - 1]);
      }
  auto al = [](size_t n) { return (n + 255) & ~size_t(255); };
  const size_t se = (size_t)b->nts_e * b->nrec_e * sizeof(double), sr = (size_t)b->nts_r * b->nrec_r * sizeof(double);
  const size_t total = al(3L * ne * 4) + al(cr.size() * 4) + 2 * al(se) + 2 * al(sr) +
                       al((nts_e + nts_r + 1) * sizeof(double));
  if (hipMalloc(&b->arena, total) != hipSuccess) { delete b; return PIHM_ERR_HIP; }
  char *base = (char *)b->arena;
  b->code_e = (int32_t *)base; base += al(3L * ne * 4);
  b->code_r = (int32_t *)base; base += al(cr.size() * 4);
  b->ft_e = (double *)base; base += al(se);
  b->v_e = (double *)base; base += al(se);
  b->ft_r = (double *)base; base += al(sr);
  b->v_r = (double *)base; base += al(sr);
  b->val = (double *)base;
  bool ok = hipMemcpy(b->code_e, ce.data(), 3L * ne * 4, hipMemcpyHostToDevice) == hipSuccess &&
            hipMemcpy(b->code_r, cr.data(), cr.size() * 4, hipMemcpyHostToDevice) == hipSuccess;
  if (ok && se)
    ok = hipMemcpy(b->ft_e, ets->ftime, se, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->v_e, ets->value, se, hipMemcpyHostToDevice) == hipSuccess;
  if (ok && sr)
    ok = hipMemcpy(b->ft_r, rts->ftime, sr, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b->v_r, rts->value, sr, hipMemcpyHostToDevice) == hipSuccess;
  if (!ok) { pihm_bc_destroy(b); return PIHM_ERR_HIP; }
  *out = b;
  return PIHM_OK;
}

void pihm_bc_destroy(pihm_bc *b) {
  if (!b) return;
  if (b->arena) (void)hipFree(b->arena);
  delete b;
}

static void launch_apply(pihm_bc *b, double t) {
  pihm_ctx *c = b->ctx;
  const long n = b->n_edge + b->nr;
  const dim3 grid((unsigned)div_up(n, (long)kBlock));
  const BcSeries se{b->nrec_e, b->ft_e, b->v_e}, sr{b->nrec_r, b->ft_r, b->v_r};
  if (b->ncoded <= kBcDirect || std::isnan(t)) {   // no interval holds a NaN: the entries stay, the table may be empty
    hipLaunchKernelGGL(k_bc, grid, dim3(kBlock), 0, c->stream, b->n_edge, b->nr, b->code_e, b->code_r, se, sr, t,
                       c->args.e.ebc, c->args.r.bc);
    return;
  }
  hipLaunchKernelGGL(k_bc_interp, dim3(div_up(b->nts_e + b->nts_r, kBlock)), dim3(kBlock), 0, c->stream, b->nts_e,
                     b->nts_r, se, sr, t, b->val);
  hipLaunchKernelGGL(k_bc_scatter, grid, dim3(kBlock), 0, c->stream, b->n_edge, b->nr, b->code_e, b->code_r, b->nts_e,
                     b->val, c->args.e.ebc, c->args.r.bc);
}

int pihm_bc_apply(pihm_bc *b, double t) {
  if (!b) return PIHM_ERR_ARG;
  if (b->nts_e + b->nts_r == 0) return PIHM_OK;
  if (t < b->t_lo || t > b->t_hi) return PIHM_ERR_ARG;
  launch_apply(b, t);
  PIHM_HIP_TRY(hipGetLastError());
  return PIHM_OK;
}

int pihm_bc_time(pihm_bc *b, double t, int iters, double *ms_per_apply) {
  if (!b || iters <= 0 || !ms_per_apply || b->nts_e + b->nts_r == 0) return PIHM_ERR_ARG;
  if (t < b->t_lo || t > b->t_hi) return PIHM_ERR_ARG;
  hipEvent_t ev[2];
  for (auto &e : ev) PIHM_HIP_TRY(hipEventCreate(&e));
  PIHM_HIP_TRY(hipEventRecord(ev[0], b->ctx->stream));
  for (int it = 0; it < iters; it++) launch_apply(b, t);
  PIHM_HIP_TRY(hipGetLastError());
  PIHM_HIP_TRY(hipEventRecord(ev[1], b->ctx->stream));
  PIHM_HIP_TRY(hipEventSynchronize(ev[1]));
  float ms = 0;
  PIHM_HIP_TRY(hipEventElapsedTime(&ms, ev[0], ev[1]));
  for (auto &e : ev) (void)hipEventDestroy(e);
  *ms_per_apply = ms / iters;
  return PIHM_OK;
}

}  // extern "C"
