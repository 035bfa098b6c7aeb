// k_dyn.hip -- momentum tendencies, time step and hyperviscosity (FP64).
//
//   uv_core                 src/shared/epic_timestep.c:628-762 with the
//                           Sadourny weights of include/epic_pv_schemes.h:48-61
//   uv_drag                 src/shared/epic_timestep.c:1303-1509
//   uv_pgrad_finite_volume  src/shared/epic_timestep.c:909-1273
//   divergence_damping      src/shared/epic_subgrid.c:1792-1885
//   adams_bashforth_step    src/shared/epic_timestep.c:406-498
//   zonal/meridional hyperviscosity, d2dy2  src/shared/epic_subgrid.c:590-1232
//
// (restore_mass, src/shared/epic_adjust.c:45-96, runs inside the launches
// next to each of its calls: the advection in k_adv.hip, k_filter3 in
// k_filter.hip.)
//
// The reference carries the finite-volume faces west->east and
// south->north; here every lane recomputes the face shared with its
// neighbour with the same expression, so the result is the same bits
// without the carried dependence.
#include "kernels.h"
#include "filter_row.h"

namespace epic {

#define MEMBER const MemberDesc &d = D[mb + blockIdx.z]
#define FLAT2(j0, nJ, i0, nI)                          \
  int t_ = blockIdx.x * TPB + threadIdx.x;             \
  if (t_ >= (nJ) * (nI)) return;                       \
  const int J = (j0) + t_ / (nI);                      \
  const int I = (i0) + t_ % (nI);
// the same with the block renumbered for the XCDs (xcd_block): bx_.y and
// bx_.z stand for blockIdx.y and blockIdx.z
#define MEMBER_X                                       \
  const uint3 bx_ = xcd_block();                       \
  const MemberDesc &d = D[mb + bx_.z]
#define FLAT2_X(j0, nJ, i0, nI)                        \
  int t_ = bx_.x * TPB + threadIdx.x;                  \
  if (t_ >= (nJ) * (nI)) return;                       \
  const int J = (j0) + t_ / (nI);                      \
  const int I = (i0) + t_ % (nI);

static inline dim3 grid2(int nJ, int nI, int nK, int nm) {
  return dim3((unsigned)((nJ * nI + TPB - 1) / TPB), (unsigned)nK, (unsigned)nm);
}

// the plane the current step's tendency accumulates in: the time plane
// IT_ZERO, or the mixed mode's single FP64 plane
__device__ __forceinline__ double *cur_tend(const MemberDesc &d, double *base) {
  return d.mixed ? base : base + (size_t)d.dyn->it0 * d.N3;
}

// ------------------------------------------------------------- uv_core
// The step's first tendencies of u and v, formed (not accumulated: nothing
// before uv_core adds to them) in one launch: Coriolis and kinetic-energy
// terms with UH, VH and KIN, vertical advection, and the top sponge
// (uv_drag).  A row team (RowMap) takes one row of one plane: it forms KIN at
// its four points, filters it (the copy the u tendency takes) where the row
// lies in the filter band, and hands its neighbours over through an LDS row;
// UH, VH and the KIN of row J-1 are formed at each point that needs them, from
// u, v and H3 in cache (4 products each), and never reach memory.  As arrays
// (one launch to write them, one for each wind to read them) they and the
// cleared, read and rewritten tendencies were 9.8 GB a step at 1024x512x64 of
// which 2 GB are needed.  Marching several rows with what they share kept in
// LDS and registers was slower at nearly every size (2 rows: +1 to +3 % of the
// step, -1 % at 1024x512x64; 8 rows: +5 to +40 %): its waves wait at barriers.
// Steps before and after: FP64 256x128x20 521 and 494 us, 1024x512x64 19.1 and
// 18.7 ms; mixed, 64 members of 128x64x16, 3777 and 3630 us.
// T = float: the mixed mode's arithmetic (k_mixed.hip); the tendencies are FP64
// in both.  Plane K = 0 takes the sponge only, with its zonal pads: nothing
// after uv_drag writes its interior, whose pads the reference fills in the
// bc_lateral that ends the 3-D filter (the filter itself starts at K = 1 and
// writes the other planes').
template <class T>
struct UvPlanes {
  Plane<const double> u, v, h3;
};
// UH at point i of row j (0..nj)
template <class T>
__device__ __forceinline__ T uh_at(const MemberDesc &d, const UvPlanes<T> &p, int j, uint32_t i, int c) {
  return T(p.u.at(i, c)) * (T(.5) * (T(p.h3.at(i, c)) + T(p.h3.at(i, c - 1)))) * T(d.ninv_h[j]);
}
// VH at point i of row j; rows 0 and nj+1 are zero as in the reference's
// cleared buffers
template <class T>
__device__ __forceinline__ T vh_at(const MemberDesc &d, const UvPlanes<T> &p, int j, uint32_t i, int c) {
  if (j < 1 || j > d.nj) return T(0.);
  return T(p.v.at(i, c)) * (T(.5) * (T(p.h3.at(i, c)) + T(p.h3.at(i - d.Ia, c)))) * T(d.minv_v[j]);
}
// KIN at point i of row j (get_kin, src/shared/epic_funcs_diag.c:2694-2847)
template <class T>
__device__ __forceinline__ T kin_at(const MemberDesc &d, const UvPlanes<T> &p, int j, uint32_t i) {
  const int jj = 2 * j;
  const uint32_t in = i + d.Ia, is = i - d.Ia;
  const T mn1 = T(d.mn[jj + 1]), mi0 = T(d.mn_inv[jj]), mi2 = T(d.mn_inv[jj + 2]);
  T u2 = T(p.u[i]), u4 = T(p.u.at(i, 1)), v2 = T(p.v[i]), v4 = T(p.v[in]);
  const T kc = (u2 * u2 + u4 * u4 + mn1 * (v2 * v2 * mi0 + v4 * v4 * mi2)) * T(.25);
  if (d.pv_al81 || j == 0 || j == d.nj) return kc;
  u2 = T(.5) * (T(p.u[in]) + T(p.u[is]));
  u4 = T(.5) * (T(p.u.at(in, 1)) + T(p.u.at(is, 1)));
  v2 = T(.5) * (T(p.v.at(i, 1)) + T(p.v.at(i, -1)));
  v4 = T(.5) * (T(p.v.at(in, 1)) + T(p.v.at(in, -1)));
  const T ks = (u2 * u2 + u4 * u4 + mn1 * (v2 * v2 * mi0 + v4 * v4 * mi2)) * T(.25);
  return (T(5.) / T(6.)) * kc + (T(1.) / T(6.)) * ks;
}
template <bool WIDE, class T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_uv_core(const MemberDesc *D, int mb) {
  MEMBER;
  constexpr bool F64 = std::is_same<T, double>::value;
  extern __shared__ double lds_raw[];
  const RowMap m = row_map(d.ni);
  const int ni = d.ni, nj = d.nj, K = blockIdx.y;
  const int Jr = blockIdx.x * m.rpb + (WIDE ? __builtin_amdgcn_readfirstlane(m.g) : m.g);
  const bool live = Jr <= nj;
  const int J = live ? Jr : nj;
  const size_t o = (size_t)K * d.N2;
  const UvPlanes<T> p{{d.U + o}, {d.V + o}, {d.H3 + o}};
  const Plane<const double> us{d.USPIN + o};
  const Plane<double> du{cur_tend(d, d.DUDT) + o}, dv{cur_tend(d, d.DVDT) + o};
  const bool sponge = K <= d.k_sponge;
  const double ts = sponge ? d.t_sponge[K] : 0.;
  auto drag = [&](double x, double w) { return F64 ? x - (ts) * w : x - (double)((float)ts * (float)w); };
  if (K == 0) {  // uniform per block
    if (!live) return;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int I = 1 + m.lane + m.stride * q;
      const uint32_t i = ix2(d, J, I);
      const double x = drag(0., p.u[i] - us[i]);
      du[i] = x;
      if (I == ni) du[ix2(d, J, 0)] = x;
      if (I == 1) du[ix2(d, J, ni + 1)] = x;
      if (J < 1) continue;
      const double y = drag(0., p.v[i] - 0.);
      dv[i] = y;
      if (I == ni) dv[ix2(d, J, 0)] = y;
      if (I == 1) dv[ix2(d, J, ni + 1)] = y;
    }
    return;
  }
  const Plane<const double> pv{d.PV3 + o}, w3{d.W3 + o}, uu{d.U + o - d.N2}, ud{d.U + o + d.N2}, vu{d.V + o - d.N2},
      vd{d.V + o + d.N2};
  const bool al81 = d.pv_al81;
  T *LK = reinterpret_cast<T *>(lds_raw) + (size_t)m.g * ni;  // [I-1]: filtered KIN
  T kin[4], kf[4];
#pragma unroll
  for (int q = 0; q < 4; q++) kf[q] = kin[q] = kin_at<T>(d, p, J, ix2(d, J, 1 + m.lane + m.stride * q));
  const bool filt = live && d.rflag_h[J] != 0;
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, kf, LK, J, 0, filt, m.lane);
#pragma unroll
  for (int q = 0; q < 4; q++) LK[m.lane + m.stride * q] = kf[q];
  row_sync<WIDE>();
  if (!live) return;
  const int kk = 2 * K + 1;
  const double ds = d.sgth[kk - 2] - d.sgth[kk + 2];
  const T ds_inv = T(1. / ds);  // the mixed mode's
  // The stores wait for the last point: a store between two points keeps the
  // second one's loads behind it.
  double xu[4], xv[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const uint32_t i = ix2(d, J, 1 + m.lane + m.stride * q), in = i + d.Ia, is = i - d.Ia;
    auto PV = [&](int j, int c) { return T(pv.at(j == J ? i : j > J ? in : is, c)); };
    {
      const PvW<T> w = pv_weights_u<T>(al81, PV, J, 0);
      const T kw = LK[(m.lane + m.stride * q - 1) & (ni - 1)];
      T a = w.al * vh_at<T>(d, p, J + 1, in, 0) + w.be * vh_at<T>(d, p, J + 1, in, -1) +
            w.ga * vh_at<T>(d, p, J, i, -1) + w.de * vh_at<T>(d, p, J, i, 0);
      if (al81) {
        const uint32_t iw = (q == 0 && m.lane == 0) ? i + (ni - 1) : i - 1;  // UH's western pad is its point ni
        a = a + w.e2 * uh_at<T>(d, p, J, iw, 0) - w.e1 * uh_at<T>(d, p, J, i, 1);
      }
      double x = 0.;
      if constexpr (F64) {
        x += (a * w.coef + kw - kf[q]) * d.m[2 * J + 1];
        x -= .5 * (w3[i] + w3.at(i, -1)) * (uu[i] - ud[i]) / ds;
      } else {
        T y = (a * w.coef + (kw - kf[q])) * T(d.m[2 * J + 1]);
        y -= T(.5) * T(w3[i] + w3.at(i, -1)) * T(uu[i] - ud[i]) * ds_inv;
        x += (double)y;
      }
      if (sponge) x = drag(x, p.u[i] - us[i]);
      xu[q] = x;
    }
    if (J >= 1) {
      const PvW<T> w = pv_weights_v<T>(al81, PV, J, 0);
      T a = -w.ga * uh_at<T>(d, p, J, i, 1) - w.de * uh_at<T>(d, p, J, i, 0) - w.al * uh_at<T>(d, p, J - 1, is, 0) -
            w.be * uh_at<T>(d, p, J - 1, is, 1);
      if (al81) a = a + w.e2 * vh_at<T>(d, p, J - 1, is, 0) - w.e1 * vh_at<T>(d, p, J + 1, in, 0);
      const T ks = kin_at<T>(d, p, J - 1, is);
      double x = 0.;
      if constexpr (F64) {
        x += (a * w.coef + ks - kin[q]) * d.n[2 * J];
        x -= .5 * (w3[i] + w3[is]) * (vu[i] - vd[i]) / ds;
      } else {
        T y = (a * w.coef + (ks - kin[q])) * T(d.n[2 * J]);
        y -= T(.5) * T(w3[i] + w3[is]) * T(vu[i] - vd[i]) * ds_inv;
        x += (double)y;
      }
      if (sponge) x = drag(x, p.v[i] - 0.);
      xv[q] = x;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const uint32_t i = ix2(d, J, 1 + m.lane + m.stride * q);
    du[i] = xu[q];
    if (J >= 1) dv[i] = xv[q];
  }
}
template <class T>
static void uv_core_t(hipStream_t s, const Bucket &b) {
  const int rpb = rows_per_block(b.ni);
  ROWS_LAUNCH(b, "k_uv_core", (k_uv_core<true, T>), (k_uv_core<false, T>), dim3((b.nj + rpb) / rpb, b.nk, b.nm),
              dim3(256), sizeof(T) * rpb * b.ni, s, b.D, b.mb);
}
void L_uv_core(hipStream_t s, const Bucket &b) {
  if (b.mixed) uv_core_t<float>(s, b);
  else uv_core_t<double>(s, b);
}

// ------------------------------------------------------------- uv_drag
// t_rad (src/shared/epic_sensible_heating.c:217-314): the Held-Suarez
// cooling time, or the tabulated one at the interface pressure; the hot
// Jupiter's relaxation time is its constant tau_rad
__device__ __forceinline__ double t_rad(const MemberDesc &d, int K, int J, int I) {
  if (d.is_hj) return d.tau_rad;
  if (d.is_tab) return tab_cool_time(d, -crm_log(d.P3[ix3(d, K, J, I)]));
  const double ka = 1. / (40. * 60. * 60. * 24.), ks = 1. / (4. * 60. * 60. * 24.);
  double p = d.P3[ix3(d, K, J, I)], kt = ka, pbot = d.P3[ix3(d, d.nk, J, I)];
  double amp = (p / pbot - 0.7) / (1. - 0.7);
  if (amp > 0.) kt += (ks - ka) * d.coslat4_h[J] * amp;  // host-libm table, as the oracle
  return 1. / kt;
}

// Rayleigh drag (tau_drag, or prandtl / t_rad): one block per (K,J) row, the
// rows of u and v staged in LDS, their zonal means summed left to right as in
// the reference (the first two lanes, one wind each), then the drag on all
// lanes.  (One lane per row did it all before: 940 us of a 1354 us step at
// 128x64x20, the loads, the logarithms of t_rad and the divisions of a row
// one after another.)
__global__ void __launch_bounds__(256) k_rayleigh(const MemberDesc *D, int mb) {
  MEMBER;
  extern __shared__ double lds[];
  const int K = d.k_sponge + 1 + blockIdx.y, J = blockIdx.x, ni = d.ni;
  if (K > d.nk - 1) return;  // uniform per block, as is the next
  if (!((d.newt_cool_on && d.prandtl > 0.) || (d.tau_drag > 0. && d.tau_drag < 1.e+20))) return;
  const bool on_v = d.drag_v && J >= 1;
  const size_t row = ix3(d, K, J, 1);
  for (int i = threadIdx.x; i < ni; i += blockDim.x) {
    lds[i] = d.U[row + i];
    if (on_v) lds[ni + i] = d.V[row + i];
  }
  __syncthreads();
  double *avg = lds + 2 * ni;
  if (threadIdx.x < (on_v ? 2 : 1)) avg[threadIdx.x] = seq_acc(lds + threadIdx.x * ni, ni) / (ni);
  __syncthreads();
  double *du = cur_tend(d, d.DUDT), *dv = cur_tend(d, d.DVDT);
  const double za = (double)d.drag_zonal_avg, zb = (double)(1 - d.drag_zonal_avg);
  for (int i = threadIdx.x; i < ni; i += blockDim.x) {
    const int I = 1 + i;
    const double tr = d.newt_cool_on ? t_rad(d, K, J, I) : 0.;
    const double uray = za * avg[0] + zb * lds[i];
    const double nu0 = d.newt_cool_on ? d.prandtl / (.5 * (tr + t_rad(d, K, J, I - 1))) : 1. / d.tau_drag;
    du[row + i] -= nu0 * (uray - d.USPIN[row + i]);
    if (on_v) {
      const double vray = za * avg[1] + zb * lds[ni + i];
      const double nuv = d.newt_cool_on ? d.prandtl / (.5 * (tr + t_rad(d, K, J - 1, I))) : 1. / d.tau_drag;
      dv[row + i] -= nuv * vray;
    }
  }
}

// Held-Suarez boundary-layer drag, one lane per u- and v-column
__global__ void __launch_bounds__(256) k_hs_pbl(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 1, d.ni);
  if (!d.is_hs) return;
  const double nu00 = (1. / (24. * 60. * 60.));
  const int nk = d.nk;
  double *du = cur_tend(d, d.DUDT), *dv = cur_tend(d, d.DVDT);
  const double *P = d.P3;
  double pb = 0.5 * (P[ix3(d, nk, J, I)] + P[ix3(d, nk, J, I - 1)]);
  for (int K = nk - 1; K >= 1; K--) {
    double p3 = .5 * (P[ix3(d, K, J, I)] + P[ix3(d, K, J, I - 1)]);
    double amp = (p3 / pb - 0.7) / (1. - 0.7);
    if (amp < 0.) break;
    du[ix3(d, K, J, I)] -= nu00 * amp * d.U[ix3(d, K, J, I)];
  }
  if (J >= 1) {
    pb = 0.5 * (P[ix3(d, nk, J, I)] + P[ix3(d, nk, J - 1, I)]);
    for (int K = nk - 1; K >= 1; K--) {
      double p3 = .5 * (P[ix3(d, K, J, I)] + P[ix3(d, K, J - 1, I)]);
      double amp = (p3 / pb - 0.7) / (1. - 0.7);
      if (amp < 0.) break;
      dv[ix3(d, K, J, I)] -= nu00 * amp * d.V[ix3(d, K, J, I)];
    }
  }
}

void L_uv_drag(hipStream_t s, const Bucket &b) {
  if (b.mixed) { LM_uv_drag(s, b); return; }
  // (the top sponge is in k_uv_core)
  if (b.any_ray)
    LAUNCH(k_rayleigh, dim3(b.nj + 1, b.nk, b.nm), dim3(b.ni < 64 ? 64 : b.ni > 256 ? 256 : b.ni),
           sizeof(double) * (2 * b.ni + 2), s, b.D, b.mb);
  if (b.any_hs) LAUNCH(k_hs_pbl, grid2(b.nj + 1, b.ni, 1, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}

// ------------------------------------------------------------- pgrad
// GZ3 rows -1 and nj+1 take the zonal mean of the adjacent row, K = 0..nk:
// one wavefront per (K, pole), the row staged in LDS and summed in order
__global__ void __launch_bounds__(256) k_gz_polefill(const MemberDesc *D, int mb) {
  MEMBER;
  if (d.pgrad_trad) return;  // the traditional form reads no pole row
  extern __shared__ double row[];
  const int K = blockIdx.x >> 1, north = blockIdx.x & 1, ni = d.ni;
  const int Js = north ? d.nj : 0, Jd = north ? d.nj + 1 : -1;
  for (int i = threadIdx.x; i < ni; i += blockDim.x) row[i] = d.GZ3[ix3(d, K, Js, i + 1)];
  __syncthreads();
  if (threadIdx.x == 0) {
    double tmp = seq_acc(row, ni);
    tmp /= ni;
    row[ni] = tmp;
  }
  __syncthreads();
  const double v = row[ni];
  for (int I = threadIdx.x; I <= ni + 1; I += blockDim.x) d.GZ3[ix3(d, K, Jd, I)] = v;
}

// finite-volume pressure-gradient force.  A face of cell (K,J,I) from GZ3 on
// the levels K-1, K, K+1 of its column (C) and of the columns beside it, and P2
// above (pt) and below (pb): the corner geopotentials bottom/top, first and
// second side, the edge means b, t, and the force f.
struct PgFace {
  double b1, b2, t1, t2, b, t, pb, pt, f;
};
__device__ __forceinline__ PgFace pg_face(const double (&A)[3], const double (&C)[3], const double (&B)[3], double pt,
                                          double pb) {
  PgFace r;
  r.b1 = .25 * (C[1] + A[1] + C[2] + A[2]);
  r.b2 = .25 * (C[1] + B[1] + C[2] + B[2]);
  r.t1 = .25 * (C[1] + A[1] + C[0] + A[0]);
  r.t2 = .25 * (C[1] + B[1] + C[0] + B[0]);
  r.b = .5 * (C[1] + C[2]);
  r.t = .5 * (C[1] + C[0]);
  r.pb = pb;
  r.pt = pt;
  const double a1 = r.t2 + r.t1, b1 = r.t2 * r.t1, a2 = r.b2 + r.b1, b2 = r.b2 * r.b1;
  const double x1 = a1 * a1 - b1 - (a2 * a2 - b2), x2 = 3. * (a1 - a2);
  r.f = (-x1 * (pb - pt) + x2 * (r.t * pb - r.b * pt));
  return r;
}

// uv_pgrad_traditional (src/shared/epic_timestep.c:806-884, the reference's
// PGRAD_TRADITIONAL build): on K = 1..k_sigma-2 grad(MONT3) less the mean
// EXNER3 times grad(THETA); on K = k_sigma-1..nk-1 the h3-weighted GZ3
// difference less the p-weighted mean of the GZ3 differences of the
// interfaces above and below.  u at (K,J,I), v at J >= 1.
__device__ __forceinline__ void pgrad_traditional(const MemberDesc &d, int K, int J, int I, double *du, double *dv) {
  const double *MO = d.MONT3, *EX = d.EXNER3, *TH = d.THETA, *G = d.GZ3, *H = d.H3, *P = d.P3;
  const size_t q = ix3(d, K, J, I), w = ix3(d, K, J, I - 1), s = ix3(d, K, J - 1, I);
  if (K <= d.ks - 2) {
    du[q] -= d.m[2 * J + 1] * (MO[q] - MO[w] - .5 * (EX[q] + EX[w]) * (TH[q] - TH[w]));
    if (J >= 1) dv[q] -= d.n[2 * J] * (MO[q] - MO[s] - .5 * (EX[q] + EX[s]) * (TH[q] - TH[s]));
    return;
  }
  const size_t qu = q + d.N2, qd = q - d.N2;
  {
    const size_t wu = w + d.N2, wd = w - d.N2;
    const double hw = (G[q] * H[q] - G[w] * H[w]) * 2. / (H[q] + H[w]);
    const double up = (G[qu] + G[wu]) * (P[qu] - P[wu]) - (G[qd] + G[wd]) * (P[qd] - P[wd]);
    const double dn = P[qu] + P[wu] - P[qd] - P[wd];
    du[q] -= d.m[2 * J + 1] * (hw - up / dn);
  }
  if (J >= 1) {
    const size_t su = s + d.N2, sd = s - d.N2;
    const double hs = (G[q] * H[q] - G[s] * H[s]) * 2. / (H[q] + H[s]);
    const double up = (G[qu] + G[su]) * (P[qu] - P[su]) - (G[qd] + G[sd]) * (P[qd] - P[sd]);
    const double dn = P[qu] + P[su] - P[qd] - P[sd];
    dv[q] -= d.n[2 * J] * (hs - up / dn);
  }
}

// One lane per (K,J,I); with SROW (rows of whole wavefronts) a wavefront lies in
// one row, whose metric terms are then scalar.  GZ3 and P2 are held as columns
// of three levels, each value loaded once.
// FP64: 1198 us at 1024x512x64 with the metric terms per lane and the flat
// indices, 916 now; 256x128x20 27.5 and 20.6.  Marching 2-8 rows a lane with
// the shared face kept needs 190 VGPRs and is no faster (2 rows slower), nor
// are 128 VGPRs with spills (1390 us).
template <bool SROW>
__global__ void __launch_bounds__(256) k_pgrad(const MemberDesc *D, int mb) {
  MEMBER_X;
  const int t0 = bx_.x * TPB + threadIdx.x, Jl = t0 >> d.nlogn, K = 1 + bx_.y;
  const int J = SROW ? __builtin_amdgcn_readfirstlane(Jl) : Jl, I = 1 + (t0 & (d.ni - 1));
  if (J > d.nj) return;
  const double TOL = 1.e-2, DG = M_PI / 180.;
  if (d.pgrad_trad) {
    pgrad_traditional(d, K, J, I, cur_tend(d, d.DUDT), cur_tend(d, d.DVDT));
    return;
  }
  const size_t o = (size_t)K * d.N2;
  const uint32_t i = ix2(d, J, I), is = i - d.Ia, in = i + d.Ia;
  const Plane<const double> G[3] = {{d.GZ3 + o - d.N2}, {d.GZ3 + o}, {d.GZ3 + o + d.N2}};
  const Plane<const double> P[2] = {{d.P2 + o}, {d.P2 + o + d.N2}}, rho3{d.RHO3 + o};
  const Plane<double> du{cur_tend(d, d.DUDT) + o}, dv{cur_tend(d, d.DVDT) + o};
  // rows S (J-1), C (J), N (J+1): [column I-1, I, I+1][level K-1, K, K+1]
  double S[3][3], C[3][3], N[2][3], pc[3][2];
#pragma unroll
  for (int c = 0; c < 3; c++) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      S[c][k] = G[k].at(is, c - 1);
      C[c][k] = G[k].at(i, c - 1);
      if (c < 2) N[c][k] = G[k].at(in, c - 1);
    }
#pragma unroll
    for (int k = 0; k < 2; k++) pc[c][k] = P[k].at(i, c - 1);
  }
  const double rho = rho3.at(i, 0), dln = d.lon[2 * I + 1] * DG - d.lon[2 * (I - 1) + 1] * DG;
  {
    // ---- longitudinal component at u-point (J,I)
    const double rlns = d.rln[2 * J], rlnn = d.rln[2 * J + 2];
    PgFace w = pg_face(S[0], C[0], N[0], pc[0][0], pc[0][1]), e = pg_face(S[1], C[1], N[1], pc[1][0], pc[1][1]);
    const double west = w.f / (w.t - w.b), east = e.f / (e.t - e.b);
    const double rm = .5 * (rho + rho3.at(i, -1));
    double top, bottom, a1, a2, b1, b2, t1, t2;
    a1 = e.t2 + e.t1; a2 = w.t2 + w.t1;
    t2 = 3. * (a1 - a2);
    if (fabs(2. * (e.t - w.t) / (e.t + w.t - e.b - w.b)) > TOL) {
      b1 = e.t2 * e.t1; b2 = w.t2 * w.t1;
      t1 = a1 * a1 - b1 - (a2 * a2 - b2);
      top = (-t1 * (w.pt - e.pt) + t2 * (e.t * w.pt - w.t * e.pt)) / (e.t - w.t);
    } else {
      top = .5 * (w.pt + e.pt) * t2;
    }
    a1 = e.b2 + e.b1; a2 = w.b2 + w.b1;
    t2 = 3. * (a1 - a2);
    if (fabs(2. * (e.b - w.b) / (e.t + w.t - e.b - w.b)) > TOL) {
      b1 = e.b2 * e.b1; b2 = w.b2 * w.b1;
      t1 = a1 * a1 - b1 - (a2 * a2 - b2);
      bottom = (-t1 * (w.pb - e.pb) + t2 * (e.b * w.pb - w.b * e.pb)) / (e.b - w.b);
    } else {
      bottom = .5 * (w.pb + e.pb) * t2;
    }
    double north = 0., south = 0.;
    double pgf = top - bottom + south - north + west - east;
    const double dzn = e.t2 - e.b2 + w.t2 - w.b2, dzs = e.t1 - e.b1 + w.t1 - w.b1;
    pgf /= dln * rm * (rlns * (dzs + .5 * dzn) + rlnn * (dzn + .5 * dzs));
    du[i] += pgf;
  }
  if (J < 1) return;
  __builtin_amdgcn_sched_barrier(0);  // (the parts one after the other)
  // ---- latitudinal component at v-point (J,I)
  double ps[3][2];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int k = 0; k < 2; k++) ps[c][k] = P[k].at(is, c - 1);
  const double rlnn = d.rln[2 * J + 1];
  PgFace n = pg_face(C[0], C[1], C[2], pc[1][0], pc[1][1]), fs = pg_face(S[0], S[1], S[2], ps[1][0], ps[1][1]);
  const double rlns = d.rln[2 * J - 1], lts = d.lat[2 * J - 1] * DG, ltn = d.lat[2 * J + 1] * DG;
  const double rm = .5 * (rho + rho3.at(is, 0)), rlt = d.rlt[2 * J];
  n.f = rlnn * n.f / (n.t - n.b);
  fs.f = rlns * fs.f / (fs.t - fs.b);
  double a1, a2, b1, b2, b3, t1, t2;
  // east (c = 2) and west (c = 0) edges
  auto side = [&](int c, double ta, double tb, double ba, double bb) {
    const double zb = .125 * (C[1][1] + C[c][1] + S[1][1] + S[c][1] + C[1][2] + C[c][2] + S[1][2] + S[c][2]);
    const double zt = .125 * (C[1][0] + C[c][0] + S[1][0] + S[c][0] + C[1][1] + C[c][1] + S[1][1] + S[c][1]);
    const double pb = .25 * (pc[1][1] + pc[c][1] + ps[1][1] + ps[c][1]);
    const double pt = .25 * (pc[1][0] + pc[c][0] + ps[1][0] + ps[c][0]);
    const double x1 = ta + tb, y1 = ta * tb, x2 = ba + bb, y2 = ba * bb;
    const double u1 = x1 * x1 - y1 - (x2 * x2 - y2), u2 = 3. * (x1 - x2);
    return .5 * (rlns - rlnn) * (-u1 * (pb - pt) + u2 * (zt * pb - zb * pt)) / (zt - zb);
  };
  const double east = side(2, n.t2, fs.t2, n.b2, fs.b2), west = side(0, n.t1, fs.t1, n.b1, fs.b1);
  double top, bottom;
  a1 = n.t2 + n.t1; a2 = fs.t2 + fs.t1;
  t2 = 3. * (a1 - a2);
  if (fabs(2. * (n.t - fs.t) / (n.t + fs.t - n.b - fs.b)) > TOL) {
    b1 = n.t2 * n.t1; b2 = fs.t2 * fs.t1; b3 = n.t2 * fs.t2 + n.t1 * fs.t1;
    t1 = a1 * a1 - b1 - (a2 * a2 - b2);
    top = .5 * ((n.pt - fs.pt) * ((rlnn + rlns) * t1 + (rlnn - rlns) * (b1 + b2 - b3)) +
                (rlnn + rlns) * t2 * (n.t * fs.pt - fs.t * n.pt)) / (n.t - fs.t);
  } else {
    top = .25 * (rlnn + rlns) * (fs.pt + n.pt) * t2;
  }
  a1 = n.b2 + n.b1; a2 = fs.b2 + fs.b1;
  t2 = 3. * (a1 - a2);
  if (fabs(2. * (n.b - fs.b) / (n.t + fs.t - n.b - fs.b)) > TOL) {
    b1 = n.b2 * n.b1; b2 = fs.b2 * fs.b1; b3 = n.b2 * fs.b2 + n.b1 * fs.b1;
    t1 = a1 * a1 - b1 - (a2 * a2 - b2);
    bottom = .5 * ((n.pb - fs.pb) * ((rlnn + rlns) * t1 + (rlnn - rlns) * (b1 + b2 - b3)) +
                   (rlnn + rlns) * t2 * (n.b * fs.pb - fs.b * n.pb)) / (n.b - fs.b);
  } else {
    bottom = .25 * (rlnn + rlns) * (fs.pb + n.pb) * t2;
  }
  double pgf = top - bottom + fs.f - (n.f + west + east);
  const double dzn = n.t2 - n.b2 + n.t1 - n.b1, dzs = fs.t2 - fs.b2 + fs.t1 - fs.b1;
  pgf /= (ltn - lts) * rm * rlt * (rlns * (dzs + .5 * dzn) + rlnn * (dzn + .5 * dzs));
  dv[i] += pgf;
}

void L_pgrad(hipStream_t s, const Bucket &b) {
  LAUNCH(k_gz_polefill, dim3(2 * (b.nk + 1), 1, b.nm), dim3(64), sizeof(double) * (b.ni + 1), s, b.D, b.mb);
  // FP64 in both precision modes (k_mixed.hip says why)
  const dim3 g = grid2(b.nj + 1, b.ni, b.nk - 1, b.nm);
  if (b.ni >= 64) LAUNCH_AS("k_pgrad", k_pgrad<true>, g, dim3(TPB), 0, s, b.D, b.mb);
  else LAUNCH_AS("k_pgrad", k_pgrad<false>, g, dim3(TPB), 0, s, b.D, b.mb);
}

// ------------------------------------------------------ divergence damping
__global__ void __launch_bounds__(256) k_divdamp(const MemberDesc *D, int mb) {
  MEMBER_X;
  FLAT2_X(0, d.nj + 1, 1, d.ni);
  const int K = 1 + bx_.y;
  if (d.nudiv == 0.) return;
  const Plane<const double> div{d.sB + (size_t)K * d.N2};
  double *du = cur_tend(d, d.DUDT), *dv = cur_tend(d, d.DVDT);
  double coef = (d.lat[2 * J + 1] > 45.) ? d.nudiv * d.m0z : d.nudiv * d.m[2 * J + 1];
  du[ix3(d, K, J, I)] += coef * (div[ix2(d, J, I)] - div[ix2(d, J, I - 1)]);
  if (J >= 1) {
    double cv = d.nudiv * d.n[2 * J];
    dv[ix3(d, K, J, I)] += cv * (div[ix2(d, J, I)] - div[ix2(d, J - 1, I)]);
  }
}
void L_divdamp(hipStream_t s, const Bucket &b) {
  L_divergence(s, b, F_U, F_V, F_SB, 1, b.nk - 1);  // U filtered row by row inside
  if (b.mixed) { LM_divdamp_apply(s, b); return; }
  LAUNCH(k_divdamp, grid2(b.nj + 1, b.ni, b.nk - 1, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}

// ------------------------------------------------------ Adams-Bashforth
// Coefficients from the start-up flags of the older planes (FLOAT_MAX; the
// mixed mode's FP32 planes hold FP32's largest value), tested per wind at
// (KLO, jlo, ILO) as the reference does (jlo: u 0, v 1).
struct AbCoef {
  double c0, c1, c2;
};
template <class H>
__device__ __forceinline__ AbCoef ab_coef(const MemberDesc &d, const MemberDyn &dy, const H *hist, int jlo, H flag) {
  const size_t q = ix3(d, 1, jlo, 1);
  if (hist[(size_t)dy.itm2 * d.N3 + q] != flag) return {23. / 12., -16. / 12., 5. / 12.};
  if (hist[(size_t)dy.itm1 * d.N3 + q] != flag) return {3. / 2., -1. / 2., 0.};
  return {1., 0., 0.};
}
// the wind w (0 u, 1 v) of cell i of plane K after the step, from its value x;
// o: the plane's offset.  MIXED: FP64 accumulation of the current tendency and
// the FP32 history planes; the current tendency is then stored, rounded, in
// the history slot IT_ZERO, which the rotation at the end of the step makes
// IT_MINUS1.
template <bool MIXED>
__device__ __forceinline__ double ab_wind(const MemberDesc &d, const MemberDyn &dy, int w, size_t o, uint32_t i, double x,
                                          bool upd) {
  if constexpr (MIXED) {
    float *hist = w ? d.DVDTf : d.DUDTf;
    const AbCoef ab = ab_coef<float>(d, dy, hist, w, 3.40282347e+38f);
    const double t0 = Plane<const double>{(w ? d.DVDT : d.DUDT) + o}[i];
    if (upd) {
      const Plane<const float> h1{hist + (size_t)dy.itm1 * d.N3 + o}, h2{hist + (size_t)dy.itm2 * d.N3 + o};
      const double t1 = (ab.c1 != 0.) ? h1[i] : 0., t2 = (ab.c2 != 0.) ? h2[i] : 0.;
      x += d.dt * (ab.c0 * t0 + ab.c1 * t1 + ab.c2 * t2);
    }
    Plane<float>{hist + (size_t)dy.it0 * d.N3 + o}[i] = (float)t0;
  } else if (upd) {
    const double *tb = w ? d.DVDT : d.DUDT;
    const AbCoef ab = ab_coef<double>(d, dy, tb, w, 1.7976931348623157e308);
    const Plane<const double> h0{tb + (size_t)dy.it0 * d.N3 + o}, h1{tb + (size_t)dy.itm1 * d.N3 + o},
        h2{tb + (size_t)dy.itm2 * d.N3 + o};
    x += d.dt * (ab.c0 * h0[i] + ab.c1 * h1[i] + ab.c2 * h2[i]);
  }
  return x;
}
// TO_FIELD: the update alone, to the field with its pads.  Else to copy 1 (u)
// and 2 (v) of sD, from where k_hv4 takes it; the fields still hold the winds
// of before, and the same launch (planes 1..nk, the wind on 1..nk-1) finishes
// DZDT3, which reads them at the cell's neighbours.  (The two as launches of
// their own were 490 + 485 us at 1024x512x64 FP64, 10.5 + 11 at 256x128x20;
// together
// 867 and 16.9.)
template <bool MIXED, bool TO_FIELD>
__global__ void __launch_bounds__(256) k_ab(const MemberDesc *D, int mb) {
  MEMBER_X;
  FLAT2_X(0, d.nj + 1, 1, d.ni);
  const int K = 1 + bx_.y;
  const size_t o = (size_t)K * d.N2;
  const uint32_t i = ix2(d, J, I);
  const MemberDyn dy = *d.dyn;
  if (TO_FIELD || K < d.nk) {
#pragma unroll
    for (int w = 0; w < 2; w++) {
      double *val = w ? d.V : d.U;
      const double x = ab_wind<MIXED>(d, dy, w, o, i, Plane<const double>{val + o}[i], J >= w);
      if (J < w) continue;
      if constexpr (!TO_FIELD) {
        Plane<double>{d.sD + (size_t)(1 + w) * d.N3 + o}[i] = x;
      } else {
        const Plane<double> out{val + o};
        out[i] = x;
        // zonal pads (bc_lateral after the update)
        if (I == d.ni) out[ix2(d, J, 0)] = x;
        if (I == 1) out[ix2(d, J, d.ni + 1)] = x;
      }
    }
  }
  if constexpr (!TO_FIELD) dzdt3_at(d, K, J, I);
}
bool ab_dzdt3_fused(const Bucket &b) { return hv_fused(b); }
void L_ab(hipStream_t s, const Bucket &b) {
  const bool all = ab_dzdt3_fused(b);
  const dim3 g = grid2(b.nj + 1, b.ni, all ? b.nk : b.nk - 1, b.nm);
  if (all && b.mixed) LAUNCH_AS("k_ab<true, false>", (k_ab<true, false>), g, dim3(TPB), 0, s, b.D, b.mb);
  else if (all) LAUNCH_AS("k_ab<false, false>", (k_ab<false, false>), g, dim3(TPB), 0, s, b.D, b.mb);
  else if (b.mixed) LAUNCH_AS("k_ab<true, true>", (k_ab<true, true>), g, dim3(TPB), 0, s, b.D, b.mb);
  else LAUNCH_AS("k_ab<false, true>", (k_ab<false, true>), g, dim3(TPB), 0, s, b.D, b.mb);
}

// monotone filtered geopotential, K = nk-1 down to 0 (src/shared/epic_timestep.c:176-196)
__global__ void __launch_bounds__(256) k_gz_mono(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 0, d.ni + 2);
  double *gz = d.gz;
  double below = gz[ix3(d, d.nk, J, I)];
  // levels go eight at a time: their loads are issued together ahead of the
  // chain (each level is read before it is written; the order of the chain
  // is unchanged)
  int K = d.nk - 1;
  for (; K >= 7; K -= 8) {
    double g[8];
#pragma unroll
    for (int u = 0; u < 8; u++) g[u] = gz[ix3(d, K - u, J, I)];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      double v;
      if (fcmp_d(below, 0.) == 0) v = 1.e-3;
      else v = dmax(g[u], below + fabs(below) * 1.e-5);
      gz[ix3(d, K - u, J, I)] = v;
      below = v;
    }
  }
  for (; K >= 0; K--) {
    size_t q = ix3(d, K, J, I);
    double v;
    if (fcmp_d(below, 0.) == 0) v = 1.e-3;
    else v = dmax(gz[q], below + fabs(below) * 1.e-5);
    gz[q] = v;
    below = v;
  }
}
// gz = GZ3 with planes 0..nk-1 zonally filtered (rows of the h-grid band),
// one block per (K,J) row of the whole plane (J = -1..nj+1), pads included
template <bool WIDE>
__global__ void __launch_bounds__(256) k_gz_filtercopy(const MemberDesc *D, int mb) {
  MEMBER;
  extern __shared__ double lds[];
  const RowMap m = row_map(d.ni);
  const int Jr = (int)(blockIdx.x * m.rpb + m.g) - 1, K = blockIdx.y, ni = d.ni;
  const bool live = Jr <= d.nj + 1;
  const int J = live ? Jr : 0;
  const Plane<const double> src{d.GZ3 + (size_t)K * d.N2};
  const Plane<double> dst{d.gz + (size_t)K * d.N2};
  double v[4];
#pragma unroll
  for (int q = 0; q < 4; q++) v[q] = src[ix2(d, J, 1 + m.lane + m.stride * q)];
  // the lanes that hold points 1 and ni also move the pads
  const bool first = m.lane == 0, last = m.lane == m.stride - 1;
  double pe = 0., pw = 0.;
  if (first) pe = src[ix2(d, J, ni + 1)];
  if (last) pw = src[ix2(d, J, 0)];
  const bool filt = live && K <= d.nk - 1 && J >= 0 && J <= d.nj && d.rflag_h[J] != 0;
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, v, lds + (size_t)m.g * ni, J < 0 ? 0 : J, 0, filt, m.lane);
  if (!live) return;
#pragma unroll
  for (int q = 0; q < 4; q++) dst[ix2(d, J, 1 + m.lane + m.stride * q)] = v[q];
  if (first) dst[ix2(d, J, ni + 1)] = filt ? v[0] : pe;
  if (last) dst[ix2(d, J, 0)] = filt ? v[3] : pw;
}
void L_gz_filtercopy(hipStream_t s, const Bucket &b) {
  const int rpb = rows_per_block(b.ni);
  ROWS_LAUNCH(b, "k_gz_filtercopy", k_gz_filtercopy<true>, k_gz_filtercopy<false>, dim3((b.nj + 3 + rpb - 1) / rpb, b.nk + 2, b.nm), dim3(256), sizeof(double) * rpb * b.ni, s,
         b.D, b.mb);
}

void L_gz_mono(hipStream_t s, const Bucket &b) {
  LAUNCH(k_gz_mono, grid2(b.nj + 1, b.ni + 2, 1, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}

// ------------------------------------------------------ hyperviscosity
struct HvRange { int k0, k1, jbot, jh; };
__device__ __forceinline__ HvRange hv_range(const MemberDesc &d, int kind) {
  HvRange r;
  r.k0 = (kind == 3) ? d.ks - 1 : 1;
  r.k1 = (kind <= 1) ? d.nk - 1 : d.nk;
  r.jbot = (kind == 1) ? 1 : 0;
  r.jh = (kind == 1) ? 0 : 1;
  return r;
}

// field i of a set and its member
#define SET_MEMBER                                              \
  const int fi = (int)blockIdx.z / nm;                          \
  const MemberDesc &d = D[mb + (int)blockIdx.z - fi * nm];      \
  const int f = fs.f[fi], kind = fs.kind[fi]

// The two d2dy2 passes of del^4 (coef2, then coef4) in one launch, by
// column: a thread owns column I of a tile of TJ rows of one plane, loads
// the field on rows J0-2..J0+TJ+1 (clipped to 0..jmax) into registers at
// once (all the loads in flight together), and forms each first-pass value
// it needs from them (three per output row, rather than staging them: the
// same expressions, so the same values).  Rows 0, 1, jmax-1 and jmax, whose
// stencils are shifted, read the field again (from cache).
template <class T, int TJ>
__global__ void __launch_bounds__(256) k_d2dy2_cols(const MemberDesc *D, int mb, int nm, FieldSet fs) {
  SET_MEMBER;
  const int vg = (kind == 1);
  const int jmax = vg ? d.nj + 1 : d.nj;
  HvRange r = hv_range(d, kind);
  const int K = r.k0 + blockIdx.y;
  if (K > r.k1) return;  // uniform per block
  const int nchunk = d.ni / (int)blockDim.x, tile = blockIdx.x / nchunk, chunk = blockIdx.x - tile * nchunk;
  const int J0 = tile * TJ;
  if (J0 > jmax) return;  // uniform per block (the grid covers the v rows)
  const int I = 1 + chunk * (int)blockDim.x + (int)threadIdx.x;
  const Plane<const double> hh{fld_ptr(d, f) + (size_t)K * d.N2};
  const Plane<T> out{reinterpret_cast<T *>(d.sB.get()) + (size_t)(fs.copy0 + fi) * d.N3 + (size_t)K * d.N2};
  const double *cx = vg ? d.vcx : d.hcx, *cy = vg ? d.vcy : d.hcy, *cz = vg ? d.vcz : d.hcz;
  const T c2 = T(d.coef2), c4 = T(d.coef4);
  T w[TJ + 4];  // rows J0-2 .. J0+TJ+1
#pragma unroll
  for (int t = 0; t < TJ + 4; t++) {
    const int J = J0 - 2 + t;
    w[t] = (J >= 0 && J <= jmax) ? T(hh[ix2(d, J, I)]) : T(0.);
  }
  // first pass at row j from rows (j0, j1, j2)
  auto p1 = [&](int j, T h0, T h1, T h2) {
    T a0 = c2 * T(cx[j]), a1 = c2 * T(cy[j]), a2 = c2 * T(cz[j]);
    return a0 * h0 + a1 * h1 + a2 * h2;
  };
  auto fld = [&](int j) { return T(hh[ix2(d, j, I)]); };
  auto p1_at = [&](int j) {  // any row, stencil shifted at the ends
    const int c = min(max(j, 1), jmax - 1);
    return p1(j, fld(c - 1), fld(c), fld(c + 1));
  };
#pragma unroll
  for (int t = 0; t < TJ; t++) {
    const int J = J0 + t;
    if (J > jmax) break;
    T q0, q1, q2;
    if (J >= 2 && J <= jmax - 2) {
      q0 = p1(J - 1, w[t], w[t + 1], w[t + 2]);
      q1 = p1(J, w[t + 1], w[t + 2], w[t + 3]);
      q2 = p1(J + 1, w[t + 2], w[t + 3], w[t + 4]);
    } else {
      const int c = min(max(J, 1), jmax - 1);
      q0 = p1_at(c - 1);
      q1 = p1_at(c);
      q2 = p1_at(c + 1);
    }
    T a0 = c4 * T(cx[J]), a1 = c4 * T(cy[J]), a2 = c4 * T(cz[J]);
    out[ix2(d, J, I)] = a0 * q0 + a1 * q1 + a2 * q2;
  }
}

// Rows of the order-2(pass+1) result D (copy i of sB, or of sC when src is
// 1; 1024/ni rows per block), for a member that applies that order
// (nu > 0): D is zonally filtered in LDS (rows of the filter band), then
// A += DT*sign*D on the kind's rows (sign -1 for del^4 and del^8, +1 for
// del^6) and the zonal pads of every row 0..nj+1 are written; when a higher
// order follows, the filtered D goes back to its copy, which the next
// order's meridional second difference reads (the reference filters it in
// place, src/shared/epic_subgrid.c:960-975).  Members that do not apply
// the order leave D and A as they are.
template <bool WIDE, class T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_hv_apply(const MemberDesc *D, int mb, int nm, FieldSet fs, int pass, int src) {
  SET_MEMBER;
  extern __shared__ double lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);
  const RowMap m = row_map(d.ni);
  HvRange r = hv_range(d, kind);
  const int K = r.k0 + blockIdx.y, Jr = blockIdx.x * m.rpb + m.g;
  if (K > r.k1 || hv_nu(d, pass) == 0. || hv_passes(d) <= pass) return;  // uniform per block
  const bool live = Jr <= d.nj + 1;
  const int J = live ? Jr : 0, ni = d.ni, vg = (kind == 1);
  const Plane<double> a{fld_ptr(d, f) + (size_t)K * d.N2};
  const Plane<T> dd{reinterpret_cast<T *>((src ? d.sC : d.sB).get()) + (size_t)(fs.copy0 + fi) * d.N3 + (size_t)K * d.N2};
  const bool upd = live && J >= r.jbot && J <= d.nj;
  // the row of A and the row of D, all loads in flight together
  double v[4];
  T x[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const size_t i = ix2(d, J, 1 + m.lane + m.stride * q);
    v[q] = a[i];
    x[q] = dd[i];
  }
  const bool filt = upd && (vg ? d.rflag_v[J] : d.rflag_h[J]) != 0;
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, x, lds + (size_t)m.g * ni, J, vg, filt, m.lane);
  if (!live) return;
  const bool back = upd && hv_passes(d) > pass + 1;
  const double sign = (pass & 1) ? -1. : 1.;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    if (upd) {
      v[q] += d.dt * sign * (double)x[q];
      a[ix2(d, J, I)] = v[q];
    }
    if (back) dd[ix2(d, J, I)] = x[q];
    if (I == ni) a[ix2(d, J, 0)] = v[q];
    if (I == 1) a[ix2(d, J, ni + 1)] = v[q];
  }
}

// One meridional second difference of the hyperviscosity chain past del^4:
// order 2(pass+1) = coef * d2dy2(order 2 pass) from copy i of sB (src 0) or
// sC (src 1) into the other, for members that run that pass
template <class T>
__global__ void __launch_bounds__(256) k_d2dy2_pass(const MemberDesc *D, int mb, int nm, FieldSet fs, int pass, int src) {
  SET_MEMBER;
  const int vg = (kind == 1);
  const int jmax = vg ? d.nj + 1 : d.nj;
  HvRange r = hv_range(d, kind);
  const int K = r.k0 + blockIdx.y;
  if (K > r.k1 || hv_passes(d) <= pass) return;  // uniform per block
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (jmax + 1) * d.ni) return;
  const int J = t / d.ni, I = 1 + t - J * d.ni;
  const size_t o = (size_t)(fs.copy0 + fi) * d.N3 + (size_t)K * d.N2;
  const Plane<const T> hh{reinterpret_cast<const T *>((src ? d.sC : d.sB).get()) + o};
  const Plane<T> out{reinterpret_cast<T *>((src ? d.sB : d.sC).get()) + o};
  const double *cx = vg ? d.vcx : d.hcx, *cy = vg ? d.vcy : d.hcy, *cz = vg ? d.vcz : d.hcz;
  int j0, j1, j2;
  if (J == 0) { j0 = 0; j1 = 1; j2 = 2; }
  else if (J == jmax) { j0 = J - 2; j1 = J - 1; j2 = J; }
  else { j0 = J - 1; j1 = J; j2 = J + 1; }
  const T c = T(hv_coef(d, pass));
  const T a0 = c * T(cx[J]), a1 = c * T(cy[J]), a2 = c * T(cz[J]);
  out[ix2(d, J, I)] = a0 * hh[ix2(d, j0, I)] + a1 * hh[ix2(d, j1, I)] + a2 * hh[ix2(d, j2, I)];
}

// the two d2dy2 passes of del^4 into copy i of sB, by column tiles of up to
// 256 columns and TJ rows (the rows_d2 knob; built in: 32 rows where that
// still gives 2048 blocks, else 16 or 8)
template <class T>
static void d2dy2_del4(hipStream_t s, const Bucket &b, const FieldSet &fs) {
  bool any_v = false;
  for (int i = 0; i < fs.n; i++) any_v |= (fs.kind[i] == 1);
  // rows 0..nj (+ nj+1 on the v grid); the kernel drops rows past its kind's
  const int jrows = any_v ? b.nj + 2 : b.nj + 1;
  const int CW = b.ni < 256 ? b.ni : 256;
  const int per = (b.ni / CW) * b.nk * fs.n * b.nm;  // blocks per row tile
  const int TJ = b.knob[KN_ROWS_D2]                           ? b.knob[KN_ROWS_D2]
                 : ((jrows + 31) / 32 * per >= 2048) ? 32
                 : ((jrows + 15) / 16 * per >= 2048) ? 16
                                                     : 8;
  dim3 g((jrows + TJ - 1) / TJ * (b.ni / CW), b.nk, fs.n * b.nm);
  if (TJ == 32) LAUNCH_AS("k_d2dy2_cols<T>", (k_d2dy2_cols<T, 32>), g, dim3(CW), 0, s, b.D, b.mb, b.nm, fs);
  else if (TJ == 16) LAUNCH_AS("k_d2dy2_cols<T>", (k_d2dy2_cols<T, 16>), g, dim3(CW), 0, s, b.D, b.mb, b.nm, fs);
  else LAUNCH_AS("k_d2dy2_cols<T>", (k_d2dy2_cols<T, 8>), g, dim3(CW), 0, s, b.D, b.mb, b.nm, fs);
}

// the mixed mode forms del^4 in FP32 (the field and its update stay FP64)
template <class T>
static void merid_hv_t(hipStream_t s, const Bucket &b, const FieldSet &fs) {
  bool any_v = false;
  for (int i = 0; i < fs.n; i++) any_v |= (fs.kind[i] == 1);
  const int jrows = any_v ? b.nj + 2 : b.nj + 1;
  d2dy2_del4<T>(s, b, fs);
  const int rpb = rows_per_block(b.ni);
  const dim3 ga((b.nj + 2 + rpb - 1) / rpb, b.nk, fs.n * b.nm);
  ROWS_LAUNCH(b, "k_hv_apply<T>", (k_hv_apply<true, T>), (k_hv_apply<false, T>), ga, dim3(256), sizeof(T) * rpb * b.ni, s, b.D, b.mb, b.nm, fs, 1, 0);
  // del^6 (pass 2, into sC) and del^8 (pass 3, back into sB)
  const dim3 gp((jrows * b.ni + TPB - 1) / TPB, b.nk, fs.n * b.nm);
  for (int pass = 2; pass < b.hv_passes; pass++) {
    const int src = (pass == 2) ? 0 : 1;
    LAUNCH(k_d2dy2_pass<T>, gp, dim3(TPB), 0, s, b.D, b.mb, b.nm, fs, pass, src);
    ROWS_LAUNCH(b, "k_hv_apply<T>", (k_hv_apply<true, T>), (k_hv_apply<false, T>), ga, dim3(256), sizeof(T) * rpb * b.ni, s, b.D, b.mb, b.nm, fs, pass, 1 - src);
  }
}
void L_merid_hv(hipStream_t s, const Bucket &b, const FieldSet &fs) {
  if (b.mixed) merid_hv_t<float>(s, b, fs);
  else merid_hv_t<double>(s, b, fs);
}

// zonal hyperviscosity: a block holds RB = 4*RW consecutive (K,J) rows in
// LDS, wavefront w owning rows w + 4u (u < RW), each lane the points
// I = 1 + lane + 64q (q < NQ) of them, which stay in registers (the field is
// read and written once); the row array is rewritten with their second
// differences for the zonal means, which are sequential sums, as the reference sums them, lane r of the
// first wavefront summing row r (one chain of additions serves RB rows).
// One row array per row (not two) lets a CU hold twice the rows, i.e. run
// twice the serial chains side by side.  Rows are strided by an odd number
// of doubles so the lanes of the serial phase fall in distinct LDS banks.
// A row is its wavefront's own except to the lane that sums it: block
// barriers stand on both sides of the sums only.
// NQ > 1 means rows of exactly 64 NQ points: no point is tested against ni,
// so all of a lane's loads are in flight together (with the test each load,
// of LDS and of memory, was waited for in its own branch: 1346 -> 841 us a
// step at 1024x512x64 with the pipelined sums of seq_acc).
template <class T, int RW, int NQ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_zonal_hv(const MemberDesc *D, int mb, int nm, FieldSet fs) {
  SET_MEMBER;
  constexpr int RB = 4 * RW;
  extern __shared__ double lds_raw[];
  T *X = reinterpret_cast<T *>(lds_raw);
  const int ni = d.ni, W = ni + 2, WS = W | 1;
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  HvRange r = hv_range(d, kind);
  const int K = r.k0 + blockIdx.y;
  const int np = hv_passes(d);
  if (K > r.k1 || np == 0) return;  // uniform over the block
  T *meanv = X + (size_t)RB * WS;
  double *a = fld_ptr(d, f) + (size_t)K * d.N2;
  const int J0 = blockIdx.x * RB, jlast = d.nj + 1;
  const bool on = NQ > 1 || lane < ni;  // lane holds points of the row
  double v[RW][NQ];
  // rows past the last one take its values and are not stored
#pragma unroll
  for (int u = 0; u < RW; u++) {
    const double *row = a + ix2(d, min(J0 + wv + 4 * u, jlast), 0);
    T *x = X + (wv + 4 * u) * WS;
#pragma unroll
    for (int q = 0; q < NQ; q++) v[u][q] = on ? row[1 + lane + 64 * q] : 0.;
    if (lane < 2) x[lane ? ni + 1 : 0] = T(row[lane ? ni + 1 : 0]);
  }
  // m (or m0 poleward of LAT0) of each row; pass p's coefficient of the
  // row is (coef[2(p+1)] mm) mm, as the reference forms it
  double mm[RW];
#pragma unroll
  for (int u = 0; u < RW; u++) {
    const int Jc = min(J0 + wv + 4 * u, d.nj);  // rows past nj are never applied
    const bool taper = fabs(d.lat[2 * Jc + r.jh]) > 45.;
    mm[u] = taper ? d.m0z : d.m[2 * Jc + r.jh];
  }
#pragma unroll
  for (int u = 0; u < RW; u++)
    if (on)
#pragma unroll
      for (int q = 0; q < NQ; q++) X[(wv + 4 * u) * WS + 1 + lane + 64 * q] = T(v[u][q]);
  wave_sync();
  for (int pass = 0; pass < np; pass++) {
    const double cp = hv_coef(d, pass);
    if (on)
#pragma unroll
      for (int u = 0; u < RW; u++) {
        T *x = X + (wv + 4 * u) * WS + 1 + lane, y[NQ];
        const T dcu = T(cp * mm[u] * mm[u]);
#pragma unroll
        for (int q = 0; q < NQ; q++) y[q] = dcu * (x[64 * q - 1] - T(2.) * x[64 * q] + x[64 * q + 1]);
        wave_sync();
#pragma unroll
        for (int q = 0; q < NQ; q++) x[64 * q] = y[q];
      }
    __syncthreads();
    if (wv == 0 && lane < RB) meanv[lane] = seq_acc(X + lane * WS + 1, ni) / T(ni);
    __syncthreads();
    // every point (and the zonal pads, copies of points ni and 1) less the
    // mean; an order with nu > 0: A += DT*sign*D on the rows of the range
    // (sign -1 for del^4 and del^8, +1 for del^6)
    const bool more = pass < np - 1;
    const double sign = (pass & 1) ? -1. : 1.;
#pragma unroll
    for (int u = 0; u < RW; u++) {
      const int J = J0 + wv + 4 * u;
      const T fm = meanv[wv + 4 * u];
      T *x = X + (wv + 4 * u) * WS + 1 + lane, y[NQ];
#pragma unroll
      for (int q = 0; q < NQ; q++) y[q] = on ? x[64 * q] - fm : T(0.);
      if (more && on) {
#pragma unroll
        for (int q = 0; q < NQ; q++) x[64 * q] = y[q];
        if (1 + lane + 64 * (NQ - 1) == ni) X[(wv + 4 * u) * WS] = y[NQ - 1];
        if (lane == 0) X[(wv + 4 * u) * WS + ni + 1] = y[0];
      }
      if (hv_nu(d, pass) != 0. && J >= r.jbot && J <= d.nj) {
#pragma unroll
        for (int q = 0; q < NQ; q++) v[u][q] += d.dt * sign * (double)y[q];
      }
    }
    wave_sync();
  }
  // the rows and their pads (the last pass has nu > 0: hv_passes)
#pragma unroll
  for (int u = 0; u < RW; u++) {
    const int J = J0 + wv + 4 * u;
    if (J > jlast) break;
    double *row = a + ix2(d, J, 0);
    if (on)
#pragma unroll
      for (int q = 0; q < NQ; q++) row[1 + lane + 64 * q] = v[u][q];
    if (1 + lane + 64 * (NQ - 1) == ni) row[0] = v[u][NQ - 1];
    if (lane == 0) row[ni + 1] = v[u][0];
  }
}

// rows per block RB (4, 8 or 16) such that a lane's registers hold at most
// 16 points (RB/4 rows x ni/64 points)
static int zhv_rows(const Bucket &b) {
  const int nq = b.ni >= 64 ? b.ni / 64 : 1;
  const int rows = (b.nj + 2) * b.nk * b.nm;
  int RB = b.knob[KN_ROWS_ZHV] ? b.knob[KN_ROWS_ZHV] : (rows / 16 >= 2048) ? 16 : (rows / 8 >= 2048) ? 8 : 4;
  while (RB > 4 && RB / 4 * nq > 16) RB /= 2;
  return RB;
}
template <class T, int RW>
static void zonal_hv_rw(hipStream_t s, const Bucket &b, const FieldSet &fs, dim3 g, size_t shm) {
  switch (b.ni >= 64 ? b.ni / 64 : 1) {
    case 1: LAUNCH_AS("k_zonal_hv<T>", (k_zonal_hv<T, RW, 1>), g, dim3(256), shm, s, b.D, b.mb, b.nm, fs); break;
    case 2: LAUNCH_AS("k_zonal_hv<T>", (k_zonal_hv<T, RW, 2>), g, dim3(256), shm, s, b.D, b.mb, b.nm, fs); break;
    case 4: LAUNCH_AS("k_zonal_hv<T>", (k_zonal_hv<T, RW, 4>), g, dim3(256), shm, s, b.D, b.mb, b.nm, fs); break;
    case 8:
      if constexpr (RW <= 2) LAUNCH_AS("k_zonal_hv<T>", (k_zonal_hv<T, RW, 8>), g, dim3(256), shm, s, b.D, b.mb, b.nm, fs);
      break;
    default:
      if constexpr (RW == 1) LAUNCH_AS("k_zonal_hv<T>", (k_zonal_hv<T, 1, 16>), g, dim3(256), shm, s, b.D, b.mb, b.nm, fs);
      break;
  }
}
template <class T>
static void zonal_hv_t(hipStream_t s, const Bucket &b, const FieldSet &fs) {
  const int RB = zhv_rows(b), WS = (b.ni + 2) | 1;
  dim3 g((b.nj + 2 + RB - 1) / RB, b.nk, fs.n * b.nm);
  const size_t shm = sizeof(T) * ((size_t)RB * WS + RB);
  if (RB == 4) zonal_hv_rw<T, 1>(s, b, fs, g, shm);
  else if (RB == 8) zonal_hv_rw<T, 2>(s, b, fs, g, shm);
  else zonal_hv_rw<T, 4>(s, b, fs, g, shm);
}
void L_zonal_hv(hipStream_t s, const Bucket &b, const FieldSet &fs) {
  if (b.mixed) zonal_hv_t<float>(s, b, fs);
  else zonal_hv_t<double>(s, b, fs);
}

// Zonal mean of a row of 256 points or more in the mixed mode (FP32): the
// row's ni values are summed as 64 partial sums, partial l = y[l] + y[l+64]
// + y[l+128] + ... left to right, which then meet pairwise, l with l+32,
// then l+16, ..., l+1 (a wavefront butterfly; IEEE addition commutes, so
// every lane ends with the same sum), and the sum is divided by ni.  Called
// by every lane of a wavefront, lane l holding partial l.
__device__ __forceinline__ float mean_butterfly(float p, int ni) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) p += __shfl_xor(p, o);
  return p / float(ni);
}

// del^4 of a field set in one launch, out of place (buckets whose members'
// highest order is del^4).  A block takes 4 RW consecutive rows of one plane.
// By columns first: thread c of G = 256/min(ni, 256) groups owns the columns
// I = 1 + c + 256 q (q < CPT) of RB = 4 RW / G rows, loads them on rows
// J0-2..J0+RB+1 and forms the two meridional second differences of del^4
// (stencils shifted at rows 0 and jmax) into LDS rows.  By rows then:
// wavefront w owns RW rows, a lane their points I = 1 + lane + 64 q (q < NQ);
// it filters the rows of the filter band, applies A += DT*(-1)*D, forms the
// zonal del^4 of the updated rows (two second differences, each less its
// zonal mean) and applies that, with wavefront barriers only but around the
// FP64 sums of long rows.  Every value is formed by the same expression as in
// k_d2dy2_cols, k_hv_apply and k_zonal_hv, which members with higher orders
// take; there the field and D cross memory three times, here the field is
// read (twice by its block and on two halo rows either side, from L2) and
// written.  Zonal means: the reference's sums left to right, a lane a row,
// RW rows side by side; from 256 points on, where a wavefront has one row,
// the block's four rows side by side in one wavefront instead (MEAN_BLOCK; a
// lane a row in each wavefront took 45.7 us against 32 at 256x128x20);
// the mixed mode's order for rows of 256 points or more (mean_butterfly;
// MEAN_BFLY).
// mode HV_TO_SCRATCH: field -> copy 1+i of sD (hdry and theta, which the
// advection reads there); HV_FROM_SCRATCH: copy 1+i of sD, where the
// Adams-Bashforth update left rows jbot..nj, -> field (u and v).  The zonal
// pads of every row 0..nj+1 that the field keeps are written as copies of
// points ni and 1.
enum { HV_TO_SCRATCH = 0, HV_FROM_SCRATCH = 1 };
enum { MEAN_WAVE, MEAN_BLOCK, MEAN_BFLY };
template <class T, int NI, int RW, int MEAN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_hv4(const MemberDesc *D, int mb, int nm, FieldSet fs, int mode) {
  SET_MEMBER;
  constexpr int ni = NI, COLS = NI < 256 ? NI : 256, CPT = NI / COLS, G = 256 / COLS, ROWS = 4 * RW, RB = ROWS / G;
  constexpr int NQ = NI < 64 ? 1 : NI / 64, WS = (NI + 2) | 1, NV = RW * NI < 64 ? 1 : RW * NI / 64;
  static_assert(RB * G == ROWS, "rows split evenly over the column groups");
  extern __shared__ double lds_raw[];
  T *X = reinterpret_cast<T *>(lds_raw);
  T *meanv = X + ROWS * WS;
  int *on = reinterpret_cast<int *>(meanv + ROWS);
  const int nj = d.nj, vg = (kind == 1);
  const HvRange r = hv_range(d, kind);
  const int K = r.k0 + blockIdx.y;
  if (K > r.k1) return;  // uniform over the block
  const int np = hv_passes(d);  // 0 or 2 (uniform)
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int Jb = blockIdx.x * ROWS;
  const size_t o = (size_t)K * d.N2;
  const Plane<double> a{fld_ptr(d, f) + o}, scr{d.sD + (size_t)(1 + fi) * d.N3 + o};
  const int jmax = vg ? nj + 1 : nj;
  // whether row j is updated, and the input on row j
  auto upd = [&](int j) { return j >= r.jbot && j <= nj; };
  auto in = [&](int j, int I) { return (mode == HV_FROM_SCRATCH && upd(j)) ? scr[ix2(d, j, I)] : a[ix2(d, j, I)]; };
  const int *rflag = vg ? d.rflag_v : d.rflag_h;
  if (np) {
    int g = threadIdx.x / COLS;
    if (COLS >= 64) g = __builtin_amdgcn_readfirstlane(g);  // the rows are the wavefront's: scalar
    const int c = threadIdx.x % COLS, R0 = g * RB, J0 = Jb + R0;
    if (threadIdx.x < ROWS) on[threadIdx.x] = upd(Jb + threadIdx.x) && rflag[Jb + threadIdx.x] != 0;
    const Plane<const double> cx{vg ? d.vcx : d.hcx}, cy{vg ? d.vcy : d.hcy}, cz{vg ? d.vcz : d.hcz};
    const T c2 = T(d.coef2), c4 = T(d.coef4);
    // first pass at row j from rows (j0, j1, j2)
    auto p1 = [&](int j, T h0, T h1, T h2) {
      T a0 = c2 * T(cx[j]), a1 = c2 * T(cy[j]), a2 = c2 * T(cz[j]);
      return a0 * h0 + a1 * h1 + a2 * h2;
    };
    // D of row J, column I (point e = I-1) to LDS, where the filter wants it
    auto put = [&](int t, int e, T x) {
      const bool band = upd(J0 + t) && rflag[J0 + t] != 0;
      X[(R0 + t) * WS + (band ? rev_pos(e, d.nlogn - 1) : e)] = x;
    };
    if (J0 >= 2 && J0 + RB - 1 <= jmax - 2) {
      // every stencil centred: the first pass of rows J0-1 .. J0+RB once each
      T w[RB + 4][CPT];  // rows J0-2 .. J0+RB+1
#pragma unroll
      for (int t = 0; t < RB + 4; t++)
#pragma unroll
        for (int q = 0; q < CPT; q++) w[t][q] = T(in(J0 - 2 + t, 1 + c + 256 * q));
#pragma unroll
      for (int q = 0; q < CPT; q++) {
        T P[RB + 2];
#pragma unroll
        for (int t = 0; t < RB + 2; t++) P[t] = p1(J0 - 1 + t, w[t][q], w[t + 1][q], w[t + 2][q]);
#pragma unroll
        for (int t = 0; t < RB; t++) {
          const int J = J0 + t;
          const T a0 = c4 * T(cx[J]), a1 = c4 * T(cy[J]), a2 = c4 * T(cz[J]);
          put(t, c + 256 * q, a0 * P[t] + a1 * P[t + 1] + a2 * P[t + 2]);
        }
      }
    } else {
      // the stencil shifted at rows 0 and jmax (both passes)
      auto p1_at = [&](int j, int I) {
        const int m = min(max(j, 1), jmax - 1);
        return p1(j, T(in(m - 1, I)), T(in(m, I)), T(in(m + 1, I)));
      };
#pragma unroll 1
      for (int t = 0; t < RB; t++) {
        const int J = J0 + t, m = min(max(J, 1), jmax - 1);
        if (J > jmax) break;
        const T a0 = c4 * T(cx[J]), a1 = c4 * T(cy[J]), a2 = c4 * T(cz[J]);
#pragma unroll 1
        for (int q = 0; q < CPT; q++) {
          const int I = 1 + c + 256 * q;
          put(t, I - 1, a0 * p1_at(m - 1, I) + a1 * p1_at(m, I) + a2 * p1_at(m + 1, I));
        }
      }
    }
  }
  // by rows: row Jb + wv*RW + u in LDS at X + (wv*RW + u)*WS
  const int R0 = wv * RW, Jw = Jb + R0;
  T *Xw = X + R0 * WS;
  const bool has = NI >= 64 || lane < NI;  // lane holds points of the row
  double v[RW][NQ];
#pragma unroll
  for (int u = 0; u < RW; u++)
#pragma unroll
    for (int q = 0; q < NQ; q++) v[u][q] = (has && upd(Jw + u)) ? in(Jw + u, 1 + lane + 64 * q) : 0.;
  if (np) {
    __syncthreads();
    bool band = false;
#pragma unroll
    for (int u = 0; u < RW; u++) band |= on[R0 + u] != 0;
    if (band) filter_wave<T, NV>(d, Xw, WS, RW, on + R0, Jw, vg, lane);
    const double sign = -1.;  // del^4
#pragma unroll
    for (int u = 0; u < RW; u++) {
      T *x = Xw + u * WS;
      const T sc = on[R0 + u] ? T(2. / (ni)) : T(1.);
      if (upd(Jw + u))
#pragma unroll
        for (int q = 0; q < NQ; q++)
          if (has) v[u][q] += d.dt * sign * (double)(on[R0 + u] ? x[swz_val(lane + 64 * q)] * sc : x[lane + 64 * q]);
    }
    wave_sync();
#pragma unroll
    for (int u = 0; u < RW; u++)
      if (has) {
        T *x = Xw + u * WS;
#pragma unroll
        for (int q = 0; q < NQ; q++) x[1 + lane + 64 * q] = T(v[u][q]);
        if (1 + lane + 64 * (NQ - 1) == ni) x[0] = T(v[u][NQ - 1]);
        if (lane == 0) x[ni + 1] = T(v[u][0]);
      }
    wave_sync();
#pragma unroll 1
    for (int pass = 0; pass < 2; pass++) {
      T part[RW];
#pragma unroll
      for (int u = 0; u < RW; u++) {
        // m (or m0 poleward of LAT0) of the row; the pass's coefficient is
        // (coef[2(p+1)] mm) mm, as the reference forms it
        const int Jc = min(Jw + u, nj);
        const double mm = fabs(d.lat[2 * Jc + r.jh]) > 45. ? d.m0z : d.m[2 * Jc + r.jh];
        const T dcu = T(hv_coef(d, pass) * mm * mm);
        T *x = Xw + u * WS + 1 + lane, y[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q++) y[q] = has ? dcu * (x[64 * q - 1] - T(2.) * x[64 * q] + x[64 * q + 1]) : T(0.);
        wave_sync();
        part[u] = y[0];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          if (has) x[64 * q] = y[q];
          if (q > 0) part[u] += y[q];
        }
      }
      if constexpr (MEAN == MEAN_BLOCK) {
        __syncthreads();
        if (threadIdx.x < ROWS) meanv[threadIdx.x] = seq_acc(X + threadIdx.x * WS + 1, ni) / T(ni);
        __syncthreads();
      } else if constexpr (MEAN == MEAN_WAVE) {
        wave_sync();
        if (lane < RW) meanv[R0 + lane] = seq_acc(Xw + lane * WS + 1, ni) / T(ni);
        wave_sync();
      }
#pragma unroll
      for (int u = 0; u < RW; u++) {
        T *x = Xw + u * WS + 1 + lane, y[NQ];
        T fm;
        if constexpr (MEAN == MEAN_BFLY) fm = mean_butterfly(part[u], ni);
        else fm = meanv[R0 + u];
#pragma unroll
        for (int q = 0; q < NQ; q++) y[q] = has ? x[64 * q] - fm : T(0.);
        if (pass == 0) {
          if (has) {
#pragma unroll
            for (int q = 0; q < NQ; q++) x[64 * q] = y[q];
            if (1 + lane + 64 * (NQ - 1) == ni) Xw[u * WS] = y[NQ - 1];
            if (lane == 0) Xw[u * WS + ni + 1] = y[0];
          }
        } else if (upd(Jw + u)) {
#pragma unroll
          for (int q = 0; q < NQ; q++) v[u][q] += d.dt * sign * (double)y[q];
        }
      }
      wave_sync();
    }
  }
#pragma unroll
  for (int u = 0; u < RW; u++) {
    const int J = Jw + u;
    if (upd(J)) {
      const Plane<double> out{mode == HV_FROM_SCRATCH ? a.p : scr.p};
      if (has) {
#pragma unroll
        for (int q = 0; q < NQ; q++) out[ix2(d, J, 1 + lane + 64 * q)] = v[u][q];
        if (mode == HV_FROM_SCRATCH) {
          if (1 + lane + 64 * (NQ - 1) == ni) a[ix2(d, J, 0)] = v[u][NQ - 1];
          if (lane == 0) a[ix2(d, J, ni + 1)] = v[u][0];
        }
      }
    } else if (np && J <= nj + 1 && lane == 0) {
      // rows the update leaves alone: their pads
      a[ix2(d, J, 0)] = a[ix2(d, J, ni)];
      a[ix2(d, J, ni + 1)] = a[ix2(d, J, 1)];
    }
  }
}

template <class T, int NI, int RW, int MEAN>
static void hv4_ni(hipStream_t s, const Bucket &b, const FieldSet &fs, int mode) {
  constexpr int rows = 4 * RW, WS = (NI + 2) | 1;
  const size_t shm = sizeof(T) * (rows * WS + rows) + sizeof(int) * rows;
  LAUNCH_AS("k_hv4", (k_hv4<T, NI, RW, MEAN>), dim3((b.nj + 2 + rows - 1) / rows, b.nk, fs.n * b.nm), dim3(256), shm, s,
            b.D, b.mb, b.nm, fs, mode);
}
// whether a bucket's hyperviscosity runs as k_hv4
bool hv_fused(const Bucket &b) { return b.hv_passes == 2; }
// rows per wavefront: those that give a thread four rows of its columns
template <class T, int MEAN>
static void hv4_t(hipStream_t s, const Bucket &b, const FieldSet &fs, int mode) {
  switch (b.ni) {
    case 8: hv4_ni<T, 8, 8, MEAN_WAVE>(s, b, fs, mode); break;
    case 16: hv4_ni<T, 16, 4, MEAN_WAVE>(s, b, fs, mode); break;
    case 32: hv4_ni<T, 32, 4, MEAN_WAVE>(s, b, fs, mode); break;
    case 64: hv4_ni<T, 64, 4, MEAN_WAVE>(s, b, fs, mode); break;
    case 128: hv4_ni<T, 128, 2, MEAN_WAVE>(s, b, fs, mode); break;
    case 256: hv4_ni<T, 256, 1, MEAN>(s, b, fs, mode); break;
    case 512: hv4_ni<T, 512, 1, MEAN>(s, b, fs, mode); break;
    default: hv4_ni<T, 1024, 1, MEAN>(s, b, fs, mode); break;
  }
}
static void hv4(hipStream_t s, const Bucket &b, const FieldSet &fs, int mode) {
  if (b.mixed) hv4_t<float, MEAN_BFLY>(s, b, fs, mode);
  else hv4_t<double, MEAN_BLOCK>(s, b, fs, mode);
}

// hyperviscosity of hdry and theta, which the advection then takes from sD's
// copies 1 and 2 (hv_fused) or from the fields; and of u and v, which the
// Adams-Bashforth update left in those copies or in the fields.  A bucket
// with a member of higher order takes the separate kernels, in place.
static void hv_inplace(hipStream_t s, const Bucket &b, const FieldSet &fs) {
  L_merid_hv(s, b, fs);
  L_zonal_hv(s, b, fs);
}
void L_hv_hth(hipStream_t s, const Bucket &b) {
  const FieldSet hth = {2, {F_HDRY, F_THETA}, {2, 3}, 1};
  if (hv_fused(b)) hv4(s, b, hth, HV_TO_SCRATCH);
  else hv_inplace(s, b, hth);
}
void L_hv_uv(hipStream_t s, const Bucket &b) {
  const FieldSet uv = {2, {F_U, F_V}, {0, 1}, 0};
  if (hv_fused(b)) hv4(s, b, uv, HV_FROM_SCRATCH);
  else hv_inplace(s, b, uv);
}

}  // namespace epic
