// noahsoil.hip - the _NOAH_ build's soil-water step after each model step.
//
// Each element's soil column: Summary's FindWaterTable and CalcLatFlx
// (src/update.c:37-43), then NoahHydrol (src/noah/noah.c:57-94): the moisture
// clamps, and SmFlx with SRT, SStep, Rosr12 and AdjSmProf.  The layer arrays
// live in HBM layer-major ([k * ne + p]) so that a wavefront reads one layer of
// 64 neighbouring elements together; four wavefronts work on 64 columns (at
// most 11 layers each) in LDS.  The water table, the lateral split, the clamps
// and the solve keep the reference's operation order.  The conductivity and
// the retention curve's slope share their powers (kr_slope), which are xpow's,
// as in the RHS; the ice factor's cube is two products, and exp is the device
// library's.  At the end the step leaves in the context what the next model
// step's RHS reads: sh2o[0], fcr, nwtbl and GwTransp's share
// (src/noah/lsm_func.c:163-185) for the new water-table layer.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "../../include/pihm_noahsoil.h"
#include "common.hpp"
#include "ctx.hpp"
#include "physics.hpp"

using namespace pihm;

namespace {

constexpr int ML = PIHM_NOAH_MAXLYR;
constexpr double SH2OMIN = 0.02;   // src/include/pihm_const.h:81

struct SoilDev {
  int32_t *nsoil;
  double *sldpth, *smcmax, *frzx;               // static
  double *smc, *sh2o, *smflxv, *runoff2_lyr;    // carried, [ML * ne]
  double *satdpth;                              // [ML * ne]
  double *runoff3;                              // carried
  double *infil, *runoff2;                      // the step's MassBalance values
  double *prev;                                 // [2 * ne] the previous Summary's unsat, gw
};

// MassBalance (src/update.c:107-160) with the _NOAH_ EtExtract split of the
// fluxes evaluated at y: infiltration re-derived from the storage change since
// the previous Summary, and the subsurface runoff that CalcLatFlx spreads.
__global__ __launch_bounds__(kBlock) void k_mass_balance_noah(int ne, SoilDev s, ElemDev e, const double *y,
                                                              const double *sub, double dt) {
  const int p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= ne) return;
  const double depth = e.depth[p], area = e.area[p];
  const double u = y[ne + p], g = y[2L * ne + p];
  double soilw0 = s.prev[ne + p] + s.prev[p];
  soilw0 = (soilw0 > depth) ? depth : soilw0;
  soilw0 = (soilw0 < 0.0) ? 0.0 : soilw0;
  double soilw1 = g + u;
  soilw1 = (soilw1 > depth) ? depth : soilw1;
  soilw1 = (soilw1 < 0.0) ? 0.0 : soilw1;
  double subrunoff = 0.0;
  for (int j = 0; j < 3; j++) subrunoff += sub[(long)j * ne + p] / area;
  // EtExtract with _NOAH_ (src/hydrol.c:43-56,79-84) at the clamped groundwater
  const double gc = (g > 0.0) ? g : 0.0;
  const double edir = e.edir[p], ett = e.ett[p], gwet = e.gwet[p];
  double edir_u, edir_g;
  if (gc > depth - e.dinf[p]) { edir_u = 0.0; edir_g = edir; }
  else { edir_u = edir; edir_g = 0.0; }
  const double ett_u = (1.0 - gwet) * ett, ett_g = gwet * ett;
  double infil = (soilw1 - soilw0) * e.porosity[p] / dt + subrunoff + edir_u + edir_g + ett_u + ett_g;
  if (infil < 0.0) {
    subrunoff -= infil;
    infil = 0.0;
  }
  s.infil[p] = infil;
  s.runoff2[p] = subrunoff;
  s.prev[p] = u;
  s.prev[ne + p] = g;
}

__global__ __launch_bounds__(kBlock) void k_soil_prev(int ne, SoilDev s, const double *y) {
  const int p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= ne) return;
  s.prev[p] = y[ne + p];
  s.prev[ne + p] = y[2L * ne + p];
}

// KrFunc (src/soil.c:8-13) and the retention curve's slope dpsi/dtheta of
// WDfCnd at relative saturation f in (0, 1).  With m = 1 - 1/beta and
// A = f^(1/m), the reference's product of powers
//   (f^(-1/m) - 1)^(-m) f^(-(1/m + 1)) = ((1 - A) / A)^(-m) / (A f)
// is 1 / (A (1 - A)^m), whose (1 - A)^m is also KrFunc's: two logarithms and
// two exponentials for both instead of five of each.
__device__ __forceinline__ void kr_slope(double f, double e1, double m, double scale, double *kr, double *slope) {
  double lo, tlo;
  const double hi = ln_pos(f, &lo);
  double thi = mul_pair(e1, hi, lo, &tlo);
  const double A = exp_pair(thi, tlo);
  const double qm = xpow(1.0 - A, m);
  const double g = 1.0 - qm;
  *kr = sqrt(f) * g * g;
  *slope = scale / (A * qm);
}

// What WDfCnd (src/noah/noah.c:2813-2861) takes from the soil alone, the same
// in every layer of a column.
struct WdfSoil {
  double range, e1, m, scale, ksatv, smcmin, sicemax, vkwgt;
};

// WDfCnd: src/noah/noah.c:2813-2861
__device__ __forceinline__ void wdf_cnd(double *wdf, double *wcnd, double smc, const WdfSoil &w) {
  double factr1 = 0.05 / w.range;
  double factr2 = (smc - w.smcmin) / w.range;
  factr2 = (factr2 > 1.0 - 5.0e-4) ? 1.0 - 5.0e-4 : factr2;
  factr2 = (factr2 < 0.0 + 5.0e-4) ? 5.0e-4 : factr2;
  factr1 = (factr1 < factr2) ? factr1 : factr2;
  double satkfunc, dpsidsm;
  kr_slope(factr2, w.e1, w.m, w.scale, &satkfunc, &dpsidsm);
  *wcnd = w.ksatv * satkfunc;
  *wdf = *wcnd * dpsidsm;
  if (w.sicemax > 0.0) {
    kr_slope(factr1, w.e1, w.m, w.scale, &satkfunc, &dpsidsm);
    *wdf = w.vkwgt * *wdf + (1.0 - w.vkwgt) * dpsidsm * satkfunc * w.ksatv;
  }
}

// Block shape of the soil-water step: 64 columns (one per lane) and four
// wavefronts.  The layers' conductivities and diffusivities, two logarithms
// and two exponentials each, depend on nothing but the layer and are dealt to
// the wavefronts; the water table and the lateral split go to the last one,
// which has the fewest layers; the recurrences down and up the column then run
// in the first, from LDS, while other blocks' wavefronts fill the SIMD.
//
// What bounds it: the chain of one column, some 11 layers of dependent FP64
// divisions, and 932 B per column of memory.  Measured (us per step, 6,000 /
// 20,011 / 100,000 columns of 11 layers): 42.4 / 46.8 / 104.6 with one thread
// per column, the column in registers (316 VGPRs, one wavefront per SIMD) and
// five powers per layer; 32.5 / 37.0 / 85.2 with the powers shared; this form
// 17.8 / 22.6 / 52.0.  The compiler reserves 100 B of scratch per lane for it
// (the water table's two layer arrays and arguments); a build without any took
// 17.8 / 22.7 / 52.3.
constexpr int kSoilCols = 64, kSoilWaves = 4;

__global__ __launch_bounds__(kSoilCols * kSoilWaves, 4) void k_noah_soil(int ne, SoilDev s, ElemDev e,
                                                                         const double *y, double dt) {
  __shared__ double lsh[ML][kSoilCols];    // liquid water after the clamps
  __shared__ double lic[ML][kSoilCols];    // ice
  __shared__ double lz[ML][kSoilCols];     // layer bottoms below the surface (negative)
  __shared__ double lsat[ML][kSoilCols];   // saturated depth per layer
  __shared__ double la[ML][kSoilCols];     // diffusivity; then Rosr12's p; then the moisture
  __shared__ double lb[ML][kSoilCols];     // conductivity; then Rosr12's delta
  __shared__ double lmax[kSoilWaves][kSoilCols];
  __shared__ int ltbl[kSoilCols];
  const int lane = (int)threadIdx.x % kSoilCols, wave = (int)threadIdx.x / kSoilCols;
  const int q = blockIdx.x * kSoilCols + lane;
  const bool own = q < ne;
  const int p = own ? q : ne - 1;          // lanes past the end repeat the last column and store nothing
  const int nsoil = s.nsoil[p];
  const double smcmax = s.smcmax[p], smcmin = e.smcmin[p];
  auto at = [ne, p](double *f, int k) -> double & { return f[(long)k * ne + p]; };
  auto put = [&](double *f, int k, double v) {
    if (own) f[(long)k * ne + p] = v;
  };

  // NoahHydrol's clamps (src/noah/noah.c:74-83) and the ice of each layer
  // (SmFlx: src/noah/noah.c:1676-1679)
  double icemax = 0.0;
  for (int k = wave; k < nsoil; k += kSoilWaves) {
    double smc = at(s.smc, k), sh2o = at(s.sh2o, k);
    smc = (smc > smcmin + SH2OMIN) ? smc : smcmin + SH2OMIN;
    smc = (smc < smcmax) ? smc : smcmax;
    sh2o = (sh2o < smc) ? sh2o : smc;
    const double sice = smc - sh2o;
    lsh[k][lane] = sh2o;
    lic[k][lane] = sice;
    icemax = (sice > icemax) ? sice : icemax;
  }
  lmax[wave][lane] = icemax;
  if (wave == kSoilWaves - 1) {
    // layer depths (src/noah/lsm_func.c:150-160), FindWaterTable (:4-55;
    // Summary and NoahHydrol call it with the same arguments, src/update.c:40,
    // src/noah/noah.c:72, so once) and CalcLatFlx (:226-255; runoff2 is
    // MassBalance's subsurface runoff)
    const double gw = y[2L * ne + p];
    double sl[ML], z = 0.0, depth = 0.0;
#pragma unroll
    for (int k = 0; k < ML; k++) sl[k] = at(s.sldpth, k);
#pragma unroll
    for (int k = 0; k < ML; k++) {
      if (k < nsoil) {
        z = (k == 0) ? -sl[0] : -sl[k] + z;
        lz[k][lane] = z;
        depth += sl[k];
      }
    }
    int nwtbl = -999;
    double sat[ML];
    if (gw <= 0.0) {
      nwtbl = nsoil;
#pragma unroll
      for (int k = 0; k < ML; k++) sat[k] = (k == nsoil - 1) ? 1.0E-3 : 0.0;
    } else if (gw > depth) {
      nwtbl = 0;
#pragma unroll
      for (int k = 0; k < ML; k++) sat[k] = (k < nsoil) ? sl[k] : 0.0;
    } else {
      double dsum = 0.0;
      bool found = false;
#pragma unroll
      for (int k = ML - 1; k >= 0; k--) {
        double v = 0.0;
        if (k < nsoil && !found) {
          if (dsum + sl[k] > gw) {
            v = gw - dsum;
            nwtbl = k + 1;
            found = true;
          } else {
            v = sl[k];
            dsum += sl[k];
          }
        }
        sat[k] = v;
      }
    }
    double sattot = 0.0;
#pragma unroll
    for (int k = 0; k < ML; k++) {
      lsat[k][lane] = sat[k];
      put(s.satdpth, k, sat[k]);
      if (k < nsoil) sattot += sat[k];
    }
    const double runoff2 = s.runoff2[p];
#pragma unroll
    for (int k = 0; k < ML; k++) {
      if (sattot <= 0.0) {
        if (k == nsoil - 1) put(s.runoff2_lyr, k, runoff2);
      } else if (k < nsoil) {
        put(s.runoff2_lyr, k, sat[k] / sattot * runoff2);
      }
    }
    ltbl[lane] = nwtbl;
  }
  __syncthreads();

  const int nwtbl = ltbl[lane];
  const double sicemax = fmax(fmax(lmax[0][lane], lmax[1][lane]), fmax(lmax[2][lane], lmax[3][lane]));
  if (nwtbl != 0) {
    const double alpha = e.alpha[p], beta = e.beta[p];
    WdfSoil ws;
    ws.range = smcmax - smcmin;
    ws.e1 = beta / (beta - 1.0);
    ws.m = (beta - 1.0) / beta;
    const double expon = 1.0 - 1.0 / beta;
    ws.scale = (1.0 - expon) / alpha / expon / ws.range;
    ws.ksatv = e.ksatv[p];
    ws.smcmin = smcmin;
    ws.sicemax = sicemax;
    ws.vkwgt = 1.0;
    if (sicemax > 0.0) {
      const double i500 = 500.0 * sicemax;
      ws.vkwgt = 1.0 / (1.0 + i500 * i500 * i500);
    }
    for (int k = wave; k < nsoil - 1; k += kSoilWaves) {
      double wdf, wcnd;
      wdf_cnd(&wdf, &wcnd, lsh[k][lane], ws);
      la[k][lane] = wdf;
      lb[k][lane] = wcnd;
    }
  }
  __syncthreads();
  if (wave != 0) return;

  double fcr = e.fcr[p], top;
  if (0 == nwtbl) {
    for (int k = 0; k < nsoil; k++) {
      put(s.smc, k, smcmax);
      put(s.sh2o, k, smcmax - lic[k][lane]);
    }
    top = smcmax - lic[0][lane];
  } else {
    // SRT: src/noah/noah.c:2315-2425
    const double CVFRZ = 3.0;
    fcr = 1.0;
    if (sicemax > 0.0) {   // without ice dice is 0
      double dice = 0.0;
      for (int k = 0; k < nsoil; k++)
        dice = (k == 0) ? -lz[0][lane] * lic[0][lane] : dice + (lz[k - 1][lane] - lz[k][lane]) * lic[k][lane];
      if (dice > 1.0e-2) {
        const double acrt = CVFRZ * s.frzx[p] / dice;
        double sum = 1.0;
        const double ialp1 = (int)round(CVFRZ) - 1;
        for (int j = 1; j < ialp1 + 1; j++) {
          int kf = 1;
          for (int jj = j + 1; jj < ialp1; jj++) kf *= jj;
          sum += xpow(acrt, CVFRZ - (double)j) / (double)kf;
        }
        fcr = 1.0 - exp(-acrt) * sum;
      }
    }
    // SRT's coefficients, SStep (src/noah/noah.c:2437-2480) and the downward
    // half of Rosr12 (:1572-1620) layer by layer: la becomes p, lb delta
    const double pddum = s.infil[p];
    double wdf = la[0][lane], wcnd = lb[0][lane];
    double z0 = lz[0][lane], z1 = lz[1][lane], sh0 = lsh[0][lane], sh1 = lsh[1][lane];
    double dsmdz = (sh0 - sh1) / (-0.5 * z1);
    double ddz = 1.0 / (-0.5 * z1);
    double pk, dk;
    {
      double bi = wdf * ddz / (-z0), ci = -bi;
      double rhstt = (wdf * dsmdz + wcnd - pddum + e.edir[p] + at(e.et, 0)) / z0;
      rhstt += at(s.runoff2_lyr, 0) / z0;
      rhstt *= dt;
      bi = 1.0 + bi * dt;
      ci *= dt;
      pk = -ci / bi;
      dk = rhstt / bi;
      la[0][lane] = pk;
      lb[0][lane] = dk;
    }
    for (int k = 1; k < nsoil; k++) {
      const bool last = k == nsoil - 1;
      const double denom2 = z0 - z1;
      double wdf2 = 0.0, wcnd2 = 0.0, dsmdz2 = 0.0, ddz2 = 0.0, ci = 0.0, z2 = 0.0, sh2 = 0.0;
      if (!last) {
        z2 = lz[k + 1][lane];
        sh2 = lsh[k + 1][lane];
        const double denom = z0 - z2;
        dsmdz2 = (sh1 - sh2) / (denom * 0.5);
        wdf2 = la[k][lane];
        wcnd2 = lb[k][lane];
        ddz2 = 2.0 / denom;
        ci = -wdf2 * ddz2 / denom2;
      }
      double numer = (wdf2 * dsmdz2) + wcnd2 - (wdf * dsmdz) - wcnd + at(e.et, k);
      numer += at(s.runoff2_lyr, k);
      double rhstt = numer / (-denom2);
      double ai = -wdf * ddz / denom2;
      double bi = -(ai + ci);
      rhstt *= dt;
      ai *= dt;
      bi = 1.0 + bi * dt;
      ci = last ? 0.0 : ci * dt;
      const double inv = 1.0 / (bi + ai * pk);
      pk = -ci * inv;
      dk = (rhstt - ai * dk) * inv;
      la[k][lane] = pk;
      lb[k][lane] = dk;
      wdf = wdf2;
      wcnd = wcnd2;
      dsmdz = dsmdz2;
      ddz = ddz2;
      z0 = z1;
      z1 = z2;
      sh1 = sh2;
    }
    // the upward half of Rosr12, whose solution is added to sh2o, and
    // AdjSmProf's upward pass (src/noah/noah.c:3081-3172): la becomes sh2omid
    double wplus = 0.0, x = 0.0;
    for (int k = nsoil - 1; k >= 0; k--) {
      x = (k == nsoil - 1) ? lb[k][lane] : la[k][lane] * x + lb[k][lane];
      const double ice = lic[k][lane];
      const double ddzk = (k != 0) ? lz[k - 1][lane] - lz[k][lane] : -lz[0][lane];
      const double mid = (lsh[k][lane] + x) + wplus / ddzk;
      const double stot = mid + ice;
      double smc;
      if (stot > smcmax) {
        smc = smcmax;
        wplus = (stot - smcmax) * ddzk;
      } else {
        const double sat = lsat[k][lane], sl = at(s.sldpth, k);
        double stotmin = (sat * smcmax + (sl - sat) * (smcmin + SH2OMIN)) / sl;
        stotmin = (stotmin > smcmax) ? smcmax : stotmin;
        stotmin = (stotmin < smcmin + SH2OMIN) ? (smcmin + SH2OMIN) : stotmin;
        if (stot < stotmin) {
          smc = stotmin;
          wplus = (stot - stotmin) * ddzk;
        } else {
          smc = stot;
          wplus = 0.0;
        }
      }
      la[k][lane] = smc - ice;
    }
    // AdjSmProf's downward pass
    for (int k = 0; k < nsoil; k++) {
      const double ice = lic[k][lane];
      const double ddzk = (k != 0) ? lz[k - 1][lane] - lz[k][lane] : -lz[0][lane];
      double sh2o = la[k][lane] + wplus / ddzk;
      const double stot = sh2o + ice;
      wplus = (stot > smcmax) ? (stot - smcmax) * ddzk : 0.0;
      double smc = (stot < smcmax) ? stot : smcmax;
      smc = (smc > smcmin + SH2OMIN) ? smc : (smcmin + SH2OMIN);
      sh2o = smc - ice;
      sh2o = (sh2o > 0.0) ? sh2o : 0.0;
      put(s.smc, k, smc);
      put(s.sh2o, k, sh2o);
      la[k][lane] = sh2o;
    }
    if (own) s.runoff3[p] = wplus / dt;
    top = la[0][lane];
    // layer fluxes, bottom up (smflxv[nsoil - 1] is 0)
    double below = 0.0;
    put(s.smflxv, nsoil - 1, 0.0);
    for (int k = nsoil - 1; k >= 1; k--) {
      below = (la[k][lane] - lsh[k][lane]) * at(s.sldpth, k) / dt + at(s.runoff2_lyr, k) + at(e.et, k) + below;
      put(s.smflxv, k - 1, below);
    }
  }

  // what the next model step's RHS reads
  if (!own) return;
  e.sh2o0[p] = top;
  e.fcr[p] = fcr;
  e.nwtbl[p] = nwtbl;
  const double ett = e.ett[p];
  const int nroot = e.nroot[p];
  double g = 0.0;
  if (ett > 0.0 && nwtbl <= nroot) {
    for (int j = (nwtbl <= 0 ? 0 : nwtbl - 1); j < nroot; j++) g += at(e.et, j);
    g = g / ett;
    g = (g > 1.0) ? 1.0 : g;
    g = (g < 0.0) ? 0.0 : g;
  }
  e.gwet[p] = g;
}

}  // namespace

struct pihm_noah_soil {
  pihm_ctx *ctx;
  int ne;
  SoilDev d;
  void *arena;
  double *scratch;     // [neq + 2 nr]: fluxes evaluated at the Summary state, carried flux saved
  int started;
};

namespace pihm {
// The soil column of a soil-water step, for the Noah land-surface step that
// shares it (noahlsm.hip): device order, layer arrays layer-major.
NoahSoilView noah_soil_view(pihm_noah_soil *s) {
  NoahSoilView v;
  v.ctx = s->ctx;
  v.ne = s->ne;
  v.nsoil = s->d.nsoil;
  v.sldpth = s->d.sldpth;
  v.smcmax = s->d.smcmax;
  v.smc = s->d.smc;
  v.sh2o = s->d.sh2o;
  return v;
}
}  // namespace pihm

namespace {

// caller-order host values of one field -> device order at dst (layers: ML
// per element, element-major on the host, layer-major on the device)
int upload(pihm_noah_soil *s, double *dst, const double *src, int layers) {
  const int ne = s->ne;
  std::vector<double> h((size_t)layers * ne);
  for (int p = 0; p < ne; p++) {
    const long ci = s->ctx->perm[p];
    for (int k = 0; k < layers; k++) h[(size_t)k * ne + p] = src[ci * layers + k];
  }
  PIHM_HIP_TRY(hipMemcpyAsync(dst, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, s->ctx->stream));
  PIHM_HIP_TRY(hipStreamSynchronize(s->ctx->stream));
  return PIHM_OK;
}

template <class T>
int download(pihm_noah_soil *s, const T *src, T *dst, int layers) {
  const int ne = s->ne;
  std::vector<T> h((size_t)layers * ne);
  PIHM_HIP_TRY(hipMemcpyAsync(h.data(), src, h.size() * sizeof(T), hipMemcpyDeviceToHost, s->ctx->stream));
  PIHM_HIP_TRY(hipStreamSynchronize(s->ctx->stream));
  for (int p = 0; p < ne; p++) {
    const long ci = s->ctx->perm[p];
    for (int k = 0; k < layers; k++) dst[ci * layers + k] = h[(size_t)k * ne + p];
  }
  return PIHM_OK;
}

int launch(pihm_noah_soil *s, double dt, const double *y_dev) {
  pihm_ctx *c = s->ctx;
  hipLaunchKernelGGL(k_noah_soil, dim3(div_up(s->ne, kSoilCols)), dim3(kSoilCols * kSoilWaves), 0, c->stream, s->ne, s->d, c->args.e,
                     y_dev, dt);
  PIHM_HIP_TRY(hipGetLastError());
  return PIHM_OK;
}

}  // namespace

extern "C" {

int pihm_noah_soil_create(pihm_ctx *ctx, const pihm_noah_soil_desc *desc, pihm_noah_soil **out) {
  if (!out) return PIHM_ERR_ARG;
  *out = nullptr;
  if (!ctx || !desc || ctx->nmem != 1 || !ctx->noah) return PIHM_ERR_ARG;
  if (!desc->nsoil || !desc->sldpth || !desc->smcmax || !desc->frzx) return PIHM_ERR_ARG;
  const int ne = ctx->ne;
  for (int i = 0; i < ne; i++) {
    const int n = desc->nsoil[i];
    if (n < 2 || n > ML) return PIHM_ERR_ARG;
    for (int k = 0; k < n; k++)
      if (!(desc->sldpth[(long)i * ML + k] > 0.0)) return PIHM_ERR_ARG;
  }
  pihm_noah_soil *s = new pihm_noah_soil();
  s->ctx = ctx;
  s->ne = ne;
  SoilDev &D = s->d;
  const size_t b1 = ((size_t)ne * sizeof(double) + 255) & ~size_t(255);
  const size_t bl = ((size_t)ML * ne * sizeof(double) + 255) & ~size_t(255);
  const size_t bi = ((size_t)ne * sizeof(int32_t) + 255) & ~size_t(255);
  double **one[] = {&D.smcmax, &D.frzx, &D.runoff3, &D.infil, &D.runoff2};
  double **lay[] = {&D.sldpth, &D.smc, &D.sh2o, &D.smflxv, &D.runoff2_lyr, &D.satdpth};
  const size_t bs = ((size_t)(ctx->neq + 2L * ctx->nr + 1) * sizeof(double) + 255) & ~size_t(255);
  const size_t total = 7 * b1 + 6 * bl + bi + bs;
  if (hipMalloc(&s->arena, total) != hipSuccess) { delete s; return PIHM_ERR_HIP; }
  char *q = (char *)s->arena;
  for (auto f : one) { *f = (double *)q; q += b1; }
  D.prev = (double *)q; q += 2 * b1;
  for (auto f : lay) { *f = (double *)q; q += bl; }
  D.nsoil = (int32_t *)q; q += bi;
  s->scratch = (double *)q;
  int rc = PIHM_OK;
  if (hipMemsetAsync(s->arena, 0, total, ctx->stream) != hipSuccess) rc = PIHM_ERR_HIP;
  std::vector<int32_t> hn(ne);
  for (int p = 0; p < ne; p++) hn[p] = desc->nsoil[ctx->perm[p]];
  if (!rc && hipMemcpyAsync(D.nsoil, hn.data(), ne * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream) != hipSuccess)
    rc = PIHM_ERR_HIP;
  if (!rc && hipStreamSynchronize(ctx->stream) != hipSuccess) rc = PIHM_ERR_HIP;
  if (!rc) rc = upload(s, D.sldpth, desc->sldpth, ML);
  if (!rc) rc = upload(s, D.smcmax, desc->smcmax, 1);
  if (!rc) rc = upload(s, D.frzx, desc->frzx, 1);
  if (rc) { pihm_noah_soil_destroy(s); return rc; }
  *out = s;
  return PIHM_OK;
}

void pihm_noah_soil_destroy(pihm_noah_soil *s) {
  if (!s) return;
  if (s->arena) (void)hipFree(s->arena);
  delete s;
}

int pihm_noah_soil_set_state(pihm_noah_soil *s, const double *smc, const double *sh2o, const double *fcr) {
  if (!s || !smc || !sh2o) return PIHM_ERR_ARG;
  int rc;
  if ((rc = upload(s, s->d.smc, smc, ML))) return rc;
  if ((rc = upload(s, s->d.sh2o, sh2o, ML))) return rc;
  ElemDev &E = s->ctx->args.e;
  if (fcr && (rc = upload(s, E.fcr, fcr, 1))) return rc;
  // the RHS's top-layer water: sh2o[0] of each element
  std::vector<double> top(s->ne);
  for (int i = 0; i < s->ne; i++) top[i] = sh2o[(long)i * ML];
  return upload(s, E.sh2o0, top.data(), 1);
}

int pihm_noah_soil_get_state(pihm_noah_soil *s, double *smc, double *sh2o, double *fcr, int32_t *nwtbl,
                             double *satdpth, double *runoff2_lyr, double *smflxv, double *runoff3) {
  if (!s) return PIHM_ERR_ARG;
  const ElemDev &E = s->ctx->args.e;
  int rc = PIHM_OK;
  if (!rc && smc) rc = download(s, s->d.smc, smc, ML);
  if (!rc && sh2o) rc = download(s, s->d.sh2o, sh2o, ML);
  if (!rc && fcr) rc = download(s, (const double *)E.fcr, fcr, 1);
  if (!rc && nwtbl) rc = download(s, (const int32_t *)E.nwtbl, nwtbl, 1);
  if (!rc && satdpth) rc = download(s, s->d.satdpth, satdpth, ML);
  if (!rc && runoff2_lyr) rc = download(s, s->d.runoff2_lyr, runoff2_lyr, ML);
  if (!rc && smflxv) rc = download(s, s->d.smflxv, smflxv, ML);
  if (!rc && runoff3) rc = download(s, s->d.runoff3, runoff3, 1);
  return rc;
}

int pihm_noah_soil_step(pihm_noah_soil *s, double dt, const double *y_dev, const double *infil,
                        const double *runoff2) {
  if (!s || !y_dev || !infil || !runoff2 || !(dt > 0.0) || !s->ctx->noah) return PIHM_ERR_ARG;
  int rc;
  if ((rc = upload(s, s->d.infil, infil, 1))) return rc;
  if ((rc = upload(s, s->d.runoff2, runoff2, 1))) return rc;
  return launch(s, dt, y_dev);
}

int pihm_noah_soil_start(pihm_noah_soil *s, const double *y_dev) {
  if (!s || !y_dev) return PIHM_ERR_ARG;
  hipLaunchKernelGGL(k_soil_prev, dim3(div_up(s->ne, kBlock)), dim3(kBlock), 0, s->ctx->stream, s->ne, s->d, y_dev);
  PIHM_HIP_TRY(hipGetLastError());
  s->started = 1;
  return PIHM_OK;
}

int pihm_noah_soil_summary(pihm_noah_soil *s, double dt, const double *y_dev) {
  if (!s || !y_dev || !(dt > 0.0) || !s->ctx->noah || !s->started) return PIHM_ERR_ARG;
  pihm_ctx *c = s->ctx;
  int rc = pihm_ctx_eval_fluxes(c, y_dev, s->scratch, s->scratch + c->neq);
  if (rc) return rc;
  hipLaunchKernelGGL(k_mass_balance_noah, dim3(div_up(s->ne, kBlock)), dim3(kBlock), 0, c->stream, s->ne, s->d,
                     c->args.e, y_dev, (const double *)c->args.rec.sub, dt);
  PIHM_HIP_TRY(hipGetLastError());
  return launch(s, dt, y_dev);
}

int pihm_noah_soil_time(pihm_noah_soil *s, double dt, const double *y_dev, int iters, double *ms) {
  if (!s || !y_dev || iters < 1 || !ms || !(dt > 0.0) || !s->ctx->noah) return PIHM_ERR_ARG;
  hipStream_t st = s->ctx->stream;
  hipEvent_t ev[2];
  for (auto &e : ev) PIHM_HIP_TRY(hipEventCreate(&e));
  int rc = PIHM_OK;
  float t = 0.0f;
  if (hipEventRecord(ev[0], st) != hipSuccess) rc = PIHM_ERR_HIP;
  for (int it = 0; !rc && it < iters; it++) rc = launch(s, dt, y_dev);
  if (!rc && (hipEventRecord(ev[1], st) != hipSuccess || hipEventSynchronize(ev[1]) != hipSuccess ||
              hipEventElapsedTime(&t, ev[0], ev[1]) != hipSuccess))
    rc = PIHM_ERR_HIP;
  for (auto &e : ev) (void)hipEventDestroy(e);
  if (!rc) *ms = (double)t / iters;
  return rc;
}

}  // extern "C"
