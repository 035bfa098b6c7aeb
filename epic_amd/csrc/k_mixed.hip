// k_mixed.hip -- the momentum kernels of the mixed-precision mode.
//
// The state (u, v, h, theta), the hydrostatic diagnostics (P3, P2, GZ3,
// MONT3, RHO3, ...) and the Adams-Bashforth accumulation stay FP64; the
// Adams-Bashforth history planes of DUDT, DVDT are FP32, and these tendency
// terms are formed in FP32: Coriolis and kinetic energy (uv_core), the
// sponge and drag (uv_drag) and divergence damping.  The finite-volume
// pressure gradient is the FP64 kernel of k_dyn.hip in both modes: its face
// integrals are products of geopotential-sized numbers whose difference is
// the small force that balances Coriolis, and formed in FP32 (even on
// geopotential shifted by the cell's own value) they left u of the hot
// Jupiter at 1024x512x64 8.4e-4 (relative L2) from the FP64 run after 100
// steps against 1.1e-5 in FP64, which costs no time (both kernels wait on
// the same loads).  The terms of the current step are summed into one FP64
// plane (DUDT, DVDT hold a single plane in this mode) and rounded to FP32
// once, when the step stores it in the history: in balanced flow the v
// tendency is the small residual of the Coriolis and pressure-gradient
// terms, which an FP32 running sum would lose.  Vertical differences of u
// and v are formed in FP64 before they are rounded.  This file is selected
// per bucket when the engine runs in the mixed mode.
#include "kernels.h"
#include "filter_row.h"

namespace epic {

#define MEMBER const MemberDesc &d = D[mb + blockIdx.z]
#define FLAT2(j0, nJ, i0, nI)                          \
  int t_ = blockIdx.x * TPB + threadIdx.x;             \
  if (t_ >= (nJ) * (nI)) return;                       \
  const int J = (j0) + t_ / (nI);                      \
  const int I = (i0) + t_ % (nI);

static inline dim3 grid2(int nJ, int nI, int nK, int nm) {
  return dim3((unsigned)((nJ * nI + TPB - 1) / TPB), (unsigned)nK, (unsigned)nm);
}

// the current step's tendency plane (FP64) and the FP32 history ring
__device__ __forceinline__ double *curU(const MemberDesc &d) { return d.DUDT; }
__device__ __forceinline__ double *curV(const MemberDesc &d) { return d.DVDT; }

// ------------------------------------------------------------- uv_drag
__device__ __forceinline__ float t_rad_f(const MemberDesc &d, int K, int J, int I) {
  if (d.is_hj) return (float)d.tau_rad;
  if (d.is_tab) return (float)tab_cool_time(d, -crm_log(d.P3[ix3(d, K, J, I)]));
  const float ka = (float)(1. / (40. * 60. * 60. * 24.)), ks = (float)(1. / (4. * 60. * 60. * 24.));
  float p = (float)d.P3[ix3(d, K, J, I)], kt = ka, pbot = (float)d.P3[ix3(d, d.nk, J, I)];
  float amp = (p / pbot - 0.7f) / (1.f - 0.7f);
  if (amp > 0.f) {
    float c = cosf((float)d.lat[2 * J + 1] * (float)(M_PI / 180.));
    kt += (ks - ka) * (c * c) * (c * c) * amp;
  }
  return 1.f / kt;
}

// Rayleigh drag: one wavefront per (K,J) row, the zonal mean by a wavefront
// reduction
__global__ void __launch_bounds__(256) km_rayleigh(const MemberDesc *D, int mb) {
  MEMBER;
  if (!((d.newt_cool_on && d.prandtl > 0.) || (d.tau_drag > 0. && d.tau_drag < 1.e+20))) return;
  const int K = d.k_sponge + 1 + blockIdx.y, J = blockIdx.x;
  if (K > d.nk - 1 || J > d.nj) return;
  double *du = curU(d), *dv = curV(d);
  const int ni = d.ni, lane = threadIdx.x;
  const float za = (float)d.drag_zonal_avg, zb = (float)(1 - d.drag_zonal_avg);
  for (int w = 0; w < 2; w++) {
    if (w == 1 && !(d.drag_v && J >= 1)) break;
    const double *X = w ? d.V : d.U;
    float s = 0.f;
    for (int I = 1 + lane; I <= ni; I += 64) s += (float)X[ix3(d, K, J, I)];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    const float avg = s / (float)ni;
    for (int I = 1 + lane; I <= ni; I += 64) {
      const size_t q = ix3(d, K, J, I);
      float ray = za * avg + zb * (float)X[q];
      float nu0;
      if (d.newt_cool_on) {
        float t0 = t_rad_f(d, K, J, I), t1 = w ? t_rad_f(d, K, J - 1, I) : t_rad_f(d, K, J, I - 1);
        nu0 = (float)d.prandtl / (.5f * (t0 + t1));
      } else {
        nu0 = (float)(1. / d.tau_drag);
      }
      if (w == 0) du[q] -= (double)(nu0 * (ray - (float)d.USPIN[q]));
      else dv[q] -= (double)(nu0 * ray);
    }
  }
}

__global__ void __launch_bounds__(256) km_hs_pbl(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 1, d.ni);
  if (!d.is_hs) return;
  const float nu00 = (float)(1. / (24. * 60. * 60.));
  const int nk = d.nk;
  double *du = curU(d), *dv = curV(d);
  const double *P = d.P3;
  float pb = 0.5f * (float)(P[ix3(d, nk, J, I)] + P[ix3(d, nk, J, I - 1)]);
  for (int K = nk - 1; K >= 1; K--) {
    float p3 = .5f * (float)(P[ix3(d, K, J, I)] + P[ix3(d, K, J, I - 1)]);
    float amp = (p3 / pb - 0.7f) / (1.f - 0.7f);
    if (amp < 0.f) break;
    du[ix3(d, K, J, I)] -= (double)(nu00 * amp * (float)d.U[ix3(d, K, J, I)]);
  }
  if (J >= 1) {
    pb = 0.5f * (float)(P[ix3(d, nk, J, I)] + P[ix3(d, nk, J - 1, I)]);
    for (int K = nk - 1; K >= 1; K--) {
      float p3 = .5f * (float)(P[ix3(d, K, J, I)] + P[ix3(d, K, J - 1, I)]);
      float amp = (p3 / pb - 0.7f) / (1.f - 0.7f);
      if (amp < 0.f) break;
      dv[ix3(d, K, J, I)] -= (double)(nu00 * amp * (float)d.V[ix3(d, K, J, I)]);
    }
  }
}

// ------------------------------------------------------ divergence damping
__global__ void __launch_bounds__(256) km_divdamp(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 1, d.ni);
  const int K = 1 + blockIdx.y;
  if (d.nudiv == 0.) return;
  const Plane<const double> div{d.sB + (size_t)K * d.N2};
  double *du = curU(d), *dv = curV(d);
  float coef = (float)((d.lat[2 * J + 1] > 45.) ? d.nudiv * d.m0z : d.nudiv * d.m[2 * J + 1]);
  du[ix3(d, K, J, I)] += (double)(coef * (float)(div[ix2(d, J, I)] - div[ix2(d, J, I - 1)]));
  if (J >= 1) {
    float cv = (float)(d.nudiv * d.n[2 * J]);
    dv[ix3(d, K, J, I)] += (double)(cv * (float)(div[ix2(d, J, I)] - div[ix2(d, J - 1, I)]));
  }
}

// ------------------------------------------------------------- launchers
void LM_uv_drag(hipStream_t s, const Bucket &b) {
  if (b.any_ray) LAUNCH(km_rayleigh, dim3(b.nj + 1, b.nk, b.nm), dim3(64), 0, s, b.D, b.mb);
  if (b.any_hs) LAUNCH(km_hs_pbl, grid2(b.nj + 1, b.ni, 1, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}
void LM_divdamp_apply(hipStream_t s, const Bucket &b) {
  LAUNCH(km_divdamp, grid2(b.nj + 1, b.ni, b.nk - 1, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}

}  // namespace epic
