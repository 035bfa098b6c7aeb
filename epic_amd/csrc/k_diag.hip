// k_diag.hip -- diagnostic kernels of the EPIC step on gfx950 (FP64).
//
//   set_p2etc         src/shared/epic_funcs_diag.c:3352-3569  (column scan)
//   store_pgrad_vars  src/shared/epic_funcs_diag.c:3595-3950  (column scans)
//   gz_from_u         src/shared/epic_funcs_diag.c:4460-4610
//   calc_heating      src/shared/epic_funcs_diag.c:4793-4869 +
//                     src/shared/epic_sensible_heating.c:51-463 (Held-Suarez,
//                     and the hot Jupiter's day-night relaxation; inside the
//                     step it is formed with T3 by k_thermo)
//   calc_w            src/shared/epic_flux.c:123-335           (column scan)
//   vorticity         src/shared/epic_funcs_diag.c:4131-4445
//   divergence        src/shared/epic_funcs_diag.c:4064-4117
//
// Column work runs in column tiles (a few levels in a lane's registers, the K
// recurrences in one lane per column over LDS); zonal means stage the row in
// LDS and sum it in one lane in the reference's order.  The arithmetic of
// each expression follows the reference's operation order.
#include <algorithm>

#include "kernels.h"
#include "filter_row.h"

namespace epic {


#define MEMBER const MemberDesc &d = D[mb + blockIdx.z]
// flat (J,I) over nJ rows starting at j0 and nI columns starting at i0
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

// ------------------------------------------------------------ utilities
__global__ void __launch_bounds__(256) k_fill(const MemberDesc *D, int mb, int f, double v) {
  MEMBER;
  double *a = fld_ptr(d, f);
  size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
  size_t stride = (size_t)gridDim.x * TPB;
  for (; i < (size_t)d.N3; i += stride) a[i] = v;
}
void L_fill(hipStream_t s, const Bucket &b, int f, double v) {
  LAUNCH(k_fill, dim3(256, 1, b.nm), dim3(TPB), 0, s, b.D, b.mb, f, v);
}

// ------------------------------------------------------------ column tiles
// A block holds C consecutive (J,I) columns (J = 0..nj, I = 0..ni+1) and all
// their levels.  A lane takes one column and KC of its levels 1..nk,
// K0..K0+KC-1, in registers, with the levels around them that it needs read
// (and their logarithms formed) again; the first lane has level 0 too; the recurrences in K (pressure from the top,
// geopotential from the bottom, the running SUM_DIV) run in one lane per
// column over one array in LDS, in the reference's order, between two
// barriers.  With C = 64 a wavefront's lanes share their levels (U): what
// depends on the level alone is scalar and the tests on it are scalar
// branches.  (With the levels strided over the lanes of 32 columns, and every
// per-level value of the others read from LDS, those tables were three of
// every five vector loads and the logarithms' and quotients' operands came
// from memory up to four times.)
template <bool U>
struct Tile {
  int C, c, K0, J, I;
  bool live, scan;  // a column of the grid; runs the column's recurrence
  uint32_t i;       // the column in a plane
  __device__ __forceinline__ Tile(const MemberDesc &d, int C_, int KC) : C(C_) {
    const int g = U ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : (int)threadIdx.x / C;
    c = U ? (int)threadIdx.x & 63 : (int)threadIdx.x - g * C;
    K0 = 1 + g * KC;
    const int nI = d.ni + 2, n = (d.nj + 1) * nI, col = blockIdx.x * C + c;
    live = col < n;
    scan = g == 0;
    const int q = live ? col : n - 1;  // lanes past the last column repeat it and store nothing
    J = q / nI;
    I = q - J * nI;
    i = ix2(d, J, I);
  }
  __device__ __forceinline__ Plane<const double> at(const MemberDesc &d, const double *f, int K) const {
    return {f + (size_t)K * d.N2};
  }
};
static inline dim3 tile_grid(const Bucket &b, int C) {
  return dim3((unsigned)(((b.nj + 1) * (b.ni + 2) + C - 1) / C), 1, (unsigned)b.nm);
}
#define COLS_LAUNCH_U(name, kern, U, sh, ...)                     \
  do {                                                            \
    if ((sh).KC == 2) LAUNCH_AS(name, (kern(2, U)), __VA_ARGS__);      \
    else if ((sh).KC == 4) LAUNCH_AS(name, (kern(4, U)), __VA_ARGS__); \
    else LAUNCH_AS(name, (kern(8, U)), __VA_ARGS__);                   \
  } while (0)
#define COLS_LAUNCH(name, kern, sh, ...)                        \
  do {                                                          \
    if ((sh).C == 64) COLS_LAUNCH_U(name, kern, true, sh, __VA_ARGS__); \
    else COLS_LAUNCH_U(name, kern, false, sh, __VA_ARGS__);             \
  } while (0)

// ------------------------------------------------------------ set_p2etc
// P3 from the top down (prefix of dsgth*g*h), the sigma-region pressures,
// h = max(h_min, dp/(g dsgth)), and the layer diagnostics P2, H3, THETA2
// (and the theta of the sigma region when update_theta)
// The FULL = 0 launch then forms store_pgrad_vars' T3 and RHO3 of its
// columns.
// FULL = 1: set_p2etc(UPDATE_THETA) with P2, H3, THETA2.  FULL = 0: the
// call that follows the advection inside the step forms P3 and h (and the
// pressure-range check) only: the P2 and H3 it would form are written again
// by the step's second set_p2etc before anything reads them, so the values
// the step leaves are the same.
// T3 and RHO3 of an interface cell (return_temp and return_density with
// x_h2 = 0); pk = (p/press0)^kappa
__device__ __forceinline__ double t3_of(double th, double pk) { return th * pk; }
__device__ __forceinline__ double rho3_of(const MemberDesc &d, double p, double t) {
  const double R_GAS = 8.314472e+3;
  return p * d.mu3 / (R_GAS * t);
}
// F: the mixed mode's exp/log/pow (m_exp)
// FP64, 1024x512x64: FULL = 0 912 us before (the levels strided over a tile's
// lanes), 533 now; FULL = 1 1346 and 1114; 256x128x20: 22 and 19, 39 and 36.
template <int FULL, bool F, int KC, bool U>
__global__ void __launch_bounds__(1024) k_set_p2etc(const MemberDesc *D, int mb, int C) {
  MEMBER;
  extern __shared__ double lds[];
  const Tile<U> T(d, C, KC);
  const int nk = d.nk, ks = d.ks, K0 = T.K0;
  double *L = lds + T.c;  // [K C]: the pressure's terms, then P3
  const double g = d.g[2 * T.J + 1], zr = d.zeta1 - d.zeta0;
  double h[KC];
#pragma unroll
  for (int r = 0; r < KC; r++) h[r] = T.at(d, d.HDRY, min(K0 + r, nk))[T.i];
  if (T.scan) L[0] = T.at(d, d.P3, 0)[T.i];
#pragma unroll
  for (int r = 0; r < KC; r++) {
    const int K = K0 + r;
    if (K <= nk) L[K * C] = d.dsgth[2 * K] * g * h[r];
  }
  __syncthreads();
  // the running sum in a register, its terms read eight at a time ahead of
  // the chain
  if (T.scan) {
    double acc = L[0];
    int K = 1;
    for (; K + 7 <= nk; K += 8) {
      double t8[8];
#pragma unroll
      for (int u = 0; u < 8; u++) t8[u] = L[(K + u) * C];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        acc = acc + t8[u];
        L[(K + u) * C] = acc;
      }
    }
    for (; K <= nk; K++) {
      acc = acc + L[K * C];
      L[K * C] = acc;
    }
  }
  __syncthreads();
  const double ptop = L[0], pbot = L[nk * C], lr = m_log<F>(ptop / pbot);
  // P3 on K0-1 .. K0+KC
  double p[KC + 2];
#pragma unroll
  for (int r = 0; r < KC + 2; r++) {
    const int K = min(K0 - 1 + r, nk);
    p[r] = L[K * C];
    if (K >= ks - 1 && K < nk) p[r] = get_p_sigma_l<F>(pbot, (d.sgth[2 * K + 1] - d.zeta0) / zr, lr);
  }
  if (!T.live) return;
  auto in = [&](double *f, int K) { return T.at(d, f, K)[T.i]; };
  auto out = [&](double *f, int K, double x) { Plane<double>{f + (size_t)K * d.N2}[T.i] = x; };
  if constexpr (!FULL) {
    // P3, h and store_pgrad_vars' per-cell part (T3, RHO3)
    double th[KC], pk[KC];
#pragma unroll
    for (int r = 0; r < KC; r++) th[r] = in(d.THETA, min(K0 + r, nk));
#pragma unroll
    for (int r = 0; r < KC; r += 2)
      m_pow2<F>(p[r + 1] / d.press0, d.kappa, p[r + 2] / d.press0, d.kappa, &pk[r], &pk[r + 1]);
    if (T.scan) {
      const double t0 = t3_of(in(d.THETA, 0), m_pow<F>(ptop / d.press0, d.kappa));
      out(d.T3, 0, t0);
      out(d.RHO3, 0, rho3_of(d, ptop, t0));
    }
#pragma unroll
    for (int r = 0; r < KC; r++) {
      const int K = K0 + r;
      if (K > nk) break;
      const double a = p[r + 1], am = p[r];
      const double hl = (a - am) / (g * d.dsgth[2 * K]), t = t3_of(th[r], pk[r]);
      out(d.P3, K, a);
      out(d.HDRY, K, dmax(d.h_min[K], hl));
      if (fcmp_d(a, am) != 0 && (am < 0. || a < 0.)) atomicOr(&d.dyn->err, 2);
      out(d.T3, K, t);
      out(d.RHO3, K, rho3_of(d, a, t));
    }
  } else {
    // p^(kappa+1) of a level's interface, formed beside P2 of the level above
    const double kp1 = d.kappa + 1., ki = 1. / d.kappa;
    double pwm, pw;
    m_pow2<F>(p[0], kp1, p[1], kp1, &pwm, &pw);
    double th = 0., thm = 0.;  // theta around a level above k_sigma-1
    if (K0 <= ks - 1) thm = theta_of_sigma<F>(d, d.sgth[2 * K0 - 1], get_sigma_l<F>(pbot, p[0], lr));
    if (T.scan && ks > 1) out(d.THETA, 0, thm);
#pragma unroll
    for (int r = 0; r < KC; r++) {
      const int K = K0 + r;
      if (K > nk) break;
      const double bot = p[r + 1], top = p[r];
      // from k_sigma down, theta2 is a linear interpolation of theta against
      // sigmatheta, table ordered from the bottom interface up
      // (src/shared/epic_funcs_diag.c:3522-3562); the interval is the same in
      // every column, found once on the host by the same search
      const int kay = K >= ks ? d.t2_kay[K] : 0;
      double y0 = 0., y1 = 0.;
      if (K >= ks) y0 = in(d.THETA, nk - kay), y1 = in(d.THETA, nk - kay - 1);
      else if (K == ks - 1) y0 = in(d.THETA, K);
      double pp, pwn = 0.;
      const double x = (pw - pwm) / (kp1 * (bot - top));
      if (r + 1 < KC) m_pow2<F>(x, ki, p[r + 2], kp1, &pp, &pwn);
      else pp = m_pow<F>(x, ki);
      if (fcmp_d(bot, top) == 0) pp = .5 * (bot + top);
      else if (top < 0. || bot < 0.) { atomicOr(&d.dyn->err, 2); pp = 0.; }
      const double hl = (bot - top) / (g * d.dsgth[2 * K]);
      double h3 = hl;
      if (K < nk) {
        const int kk = 2 * K + 1;
        const double topwt = d.dsgth[kk - 1], botwt = d.dsgth[kk + 1];
        const double hl1 = (p[r + 2] - bot) / (g * d.dsgth[2 * (K + 1)]);
        h3 = (topwt * hl + botwt * hl1) / (topwt + botwt);
      }
      double th2;
      if (K < ks - 1) {
        double s3, s2;
        m_log2<F>(bot / pbot, pp / pbot, &s3, &s2);
        th = theta_of_sigma<F>(d, d.sgth[2 * K + 1], s3 / lr);
        th2 = theta_of_sigma<F>(d, d.sgth[2 * K], s2 / lr);
        out(d.THETA, K, th);
      } else if (K >= ks) {
        const double sg = d.sgth[2 * K], hh = d.t2_h[K];
        th2 = y0 + (y1 - y0) * (sg - d.sgth[2 * (nk - kay) + 1]) / hh;
      } else {
        th2 = .5 * (y0 + thm);
      }
      out(d.P3, K, bot);
      out(d.HDRY, K, dmax(d.h_min[K], hl));
      out(d.P2, K, pp);
      out(d.H3, K, h3);
      out(d.THETA2, K, th2);
      if (T.scan && r == 0) {
        out(d.P2, 0, ptop * ptop / pp);
        out(d.H3, 0, h3);
      }
      pwm = pw;
      pw = pwn;
      thm = th;
    }
  }
}
template <int FULL, bool F>
static void set_p2etc_t(hipStream_t s, const Bucket &b) {
  const ColShape sh = col_shape(b, b.knob[KN_COLS_P2ETC]);
#define K_(KC, U) k_set_p2etc<FULL, F, KC, U>
  COLS_LAUNCH(FULL ? "k_set_p2etc<1>" : "k_set_p2etc<0>", K_, sh, tile_grid(b, sh.C), dim3(sh.nt),
              col_lds(b, sh.C), s, b.D, b.mb, sh.C);
#undef K_
}
void L_set_p2etc(hipStream_t s, const Bucket &b, int update_theta) {
  if (b.mixed) update_theta ? set_p2etc_t<1, true>(s, b) : set_p2etc_t<0, true>(s, b);
  else update_theta ? set_p2etc_t<1, false>(s, b) : set_p2etc_t<0, false>(s, b);
}

// ------------------------------------------------- store_pgrad_vars parts
// T3, EXNER3, RHO3, T2, RHO2 per cell and the top values; DZDT3 <- GZ3 when
// itime > 1, DZDT3 zeroed whole while itime <= 1
// (src/shared/epic_funcs_diag.c:3674-3690).  One lane per (K,J,I), K = 0..nk.
// full = 0 (the step's first store_pgrad_vars): T3 and RHO3 only, all that
// the geopotential integration and the filtered GZ3 copy read before the
// second call writes every output again.
template <bool F = false>
__device__ __forceinline__ double hs_relax(const MemberDesc &d, int J, double p, double t, double pbot, double pk0);
template <bool F = false>
__device__ __forceinline__ double hj_relax(const MemberDesc &d, int J, int I, double p, double t, double pk);
// full = 1 also forms the Newtonian relaxation HEAT3 of calc_heating on
// K = 1..nk, J = 0..nj and the zonal pads: it reads only P3 and T3, which
// nothing changes between here and the end of the step, where the reference
// forms it, and it takes the p^kappa formed here for T3 (a pad takes the
// value of the column it copies)
// store_pgrad_vars' per-cell part with full = 1 (after the FULL set_p2etc), one
// lane per (K,J,I), K = 1..nk, J = 0..nj, I = 0..ni+1: the operands loaded
// together (a load behind a store waits for it: the fields may overlap for all
// the compiler knows) and the cell's two powers formed side by side.  The lane
// of level 1 has level 0 too, whose RHO2 it needs.  966 us at 1024x512x64 FP64
// before, 816 now; two or four levels a lane are no faster.
template <bool F>
__global__ void __launch_bounds__(256) k_thermo(const MemberDesc *D, int mb) {
  MEMBER;
  const long itime = d.dyn->itime;
  if (itime <= 1) {
    // no lane of this kernel writes DZDT3 while itime <= 1
    const size_t nthr = (size_t)gridDim.x * gridDim.y * blockDim.x;
    for (size_t i = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x; i < (size_t)d.N3;
         i += nthr)
      d.DZDT3[i] = 0.;
  }
  FLAT2(0, d.nj + 1, 0, d.ni + 2);
  const int K = 1 + (int)blockIdx.y;
  const uint32_t i = ix2(d, J, I);
  auto in = [&](const double *f, int K) { return Plane<const double>{f + (size_t)K * d.N2}[i]; };
  auto out = [&](double *f, int K, double x) { Plane<double>{f + (size_t)K * d.N2}[i] = x; };
  const double R_GAS = 8.314472e+3;
  const bool rate = itime > 1 && I >= 1 && I <= d.ni;  // DZDT3 <- GZ3
  const double p = in(d.P3, K), th = in(d.THETA, K), p2 = in(d.P2, K), th2 = in(d.THETA2, K), gz = in(d.GZ3, K);
  double pk, pk2;
  m_pow2<F>(p / d.press0, d.kappa, p2 / d.press0, d.kappa, &pk, &pk2);
  const double t = t3_of(th, pk), t2 = t3_of(th2, pk2), rho2 = p2 * d.mu2 / (R_GAS * t2);
  const double ex = d.cp * t / th, rho3 = rho3_of(d, p, t);
  if (newt_relax_on(d)) {
    double h;
    if (d.is_tab) {
      h = 0. + tab_relax(d, p, t);
    } else if (d.is_hj) {
      h = hj_relax<F>(d, J, (I == 0) ? d.ni : (I == d.ni + 1 ? 1 : I), p, t, pk);
    } else {
      const double pk0 = (d.press0 == 1000. * 100.) ? pk : m_pow<F>(p / (1000. * 100.), d.kappa);
      h = 0. + hs_relax<F>(d, J, p, t, in(d.P3, d.nk), pk0);
    }
    out(d.HEAT3, K, h);
  }
  if (rate) out(d.DZDT3, K, gz);
  out(d.T3, K, t);
  out(d.RHO3, K, rho3);
  out(d.EXNER3, K, ex);
  out(d.T2, K, t2);
  out(d.RHO2, K, rho2);
  if (K == 1) {
    const double p0 = in(d.P3, 0), th0 = in(d.THETA, 0), t0 = t3_of(th0, m_pow<F>(p0 / d.press0, d.kappa));
    const double rho0 = rho3_of(d, p0, t0);
    out(d.T3, 0, t0);
    out(d.RHO3, 0, rho0);
    out(d.EXNER3, 0, d.cp * t0 / th0);
    out(d.RHO2, 0, rho0 * rho0 / rho2);
    out(d.THETA2, 0, d.sgth[0]);
    out(d.T2, 0, t0);
  }
}
void L_thermo(hipStream_t s, const Bucket &b) {
  const dim3 g = grid2(b.nj + 1, b.ni + 2, b.nk, b.nm);
  if (b.mixed) LAUNCH_AS("k_thermo", k_thermo<true>, g, dim3(TPB), 0, s, b.D, b.mb);
  else LAUNCH_AS("k_thermo", k_thermo<false>, g, dim3(TPB), 0, s, b.D, b.mb);
}

// ------------------------------------------------------------ RI2
// Richardson number in the layers, N^2 / ((du)^2 + (dv)^2) (get_richardson
// with kk = 2K, src/shared/epic_funcs_diag.c:3066-3156; the reference forms
// dz_inv there and leaves it unused, and its v difference carries a + on
// V(K,J+1)), with get_brunt2 of a layer (:2885-3064, no smoothing:
// Drho/Dp from the interfaces above and below, the partial derivatives of
// the ideal-gas density by centred differences of 0.1 %), return_cp
// (:3311-3337: 1004 for Held-Suarez, else the centred derivative of the
// enthalpy cpr*T*rgas of x_h2 = 0) and the layer molar mass mu2.
// Store_diag computes it for J = 0..nj, I = 1..ni, K = 1..nk and applies
// bc_lateral; every other cell stays zero.
__global__ void __launch_bounds__(256) k_richardson(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 1, d.ni);
  const int K = 1 + blockIdx.y;
  const double *U = d.U, *V = d.V;
  double dudz2 = .5 * (U[ix3(d, K - 1, J, I)] + U[ix3(d, K - 1, J, I + 1)] - U[ix3(d, K, J, I)] -
                       U[ix3(d, K, J, I + 1)]);
  double dvdz2 = .5 * (V[ix3(d, K - 1, J, I)] + V[ix3(d, K - 1, J + 1, I)] - V[ix3(d, K, J, I)] +
                       V[ix3(d, K, J + 1, I)]);
  dudz2 *= dudz2;
  dvdz2 *= dvdz2;
  double ri = 1.e+6;
  if (fcmp_d(dudz2, 0.) != 0) {
    const double R_GAS = 8.314472e+3;
    const size_t q = ix3(d, K, J, I);
    const double pressure = d.P2[q], temperature = d.T2[q], density = d.RHO2[q];
    double cp;
    if (d.is_hs) {
      cp = 1004.;
    } else {
      const double dT = temperature * 1.e-6;
      double h2 = d.cpr * (temperature + dT), h1 = d.cpr * (temperature - dT);
      h2 *= d.rgas;
      h1 *= d.rgas;
      cp = (h2 - h1) / (2. * dT);
    }
    const double mu = d.mu2, deltap = 0.001 * pressure, deltaT = 0.001 * temperature;
    const double drho_dp_T = ((pressure + deltap) * mu / (R_GAS * temperature) -
                              (pressure - deltap) * mu / (R_GAS * temperature)) / (2. * deltap);
    const double drho_dT_p = (pressure * mu / (R_GAS * (temperature + deltaT)) -
                              pressure * mu / (R_GAS * (temperature - deltaT))) / (2. * deltaT);
    const double Drho_Dp = (d.RHO3[q] - d.RHO3[ix3(d, K - 1, J, I)]) / (d.P3[q] - d.P3[ix3(d, K - 1, J, I)]);
    const double g = d.g[2 * J + 1];
    const double brunt2 =
        g * g * (Drho_Dp - drho_dp_T + temperature / (cp * density * density) * drho_dT_p * drho_dT_p);
    ri = brunt2 / (dudz2 + dvdz2);
  }
  d.RI2[ix3(d, K, J, I)] = ri;
  if (I == d.ni) d.RI2[ix3(d, K, J, 0)] = ri;
  if (I == 1) d.RI2[ix3(d, K, J, d.ni + 1)] = ri;
}
void L_richardson(hipStream_t s, const Bucket &b) {
  LAUNCH(k_richardson, grid2(b.nj + 1, b.ni, b.nk, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}

// kinetic energy of a zonally uniform u row (get_kin with v = 0)
__device__ double kin_uniform(const double *mn, const double *mni, int nj, const double *u1, int J, bool al81) {
  int jj = 2 * J;
  double u2 = u1[J], u4 = u1[J], v2 = 0., v4 = 0.;
  double kc = (u2 * u2 + u4 * u4 + mn[jj + 1] * (v2 * v2 * mni[jj] + v4 * v4 * mni[jj + 2])) * .25;
  if (al81 || J == 0 || J == nj) return kc;
  u2 = .5 * (u1[J + 1] + u1[J - 1]);
  u4 = .5 * (u1[J + 1] + u1[J - 1]);
  v2 = .5 * (0. + 0.);
  v4 = .5 * (0. + 0.);
  double ks = (u2 * u2 + u4 * u4 + mn[jj + 1] * (v2 * v2 * mni[jj] + v4 * v4 * mni[jj + 2])) * .25;
  return (5. / 6.) * kc + (1. / 6.) * ks;
}

// Gas giants: GZ_SURFACE from gradient balance with the zonal-mean bottom
// wind, in two launches: the zonal means of u, p, rho on the bottom
// interface (one wavefront per row; lanes 0-2 sum in the reference's
// sequential order), the meridional integral (one block); the column
// kernel k_gz3 that must follow copies the results into GZ_SURFACE and
// PV3's plane nk+1 as it starts each column.
template <bool F>
__global__ void __launch_bounds__(256) k_gzu_means(const MemberDesc *D, int mb) {
  MEMBER;
  if (!d.is_gas) return;
  extern __shared__ double row[];
  const int J = blockIdx.x, ni = d.ni, nk = d.nk, R = d.nj + 3;
  // RHO3 of the bottom interface formed here from P3 and theta, as
  // store_pgrad_vars forms it (the same values), so that this launch need
  // not wait for the kernel that writes RHO3
  for (int i = threadIdx.x; i < ni; i += blockDim.x) {
    const size_t q = ix3(d, nk, J, i + 1);
    const double p = d.P3[q];
    row[i] = d.U[q];
    row[ni + i] = p;
    row[2 * ni + i] = rho3_of(d, p, t3_of(d.THETA[q], m_pow<F>(p / d.press0, d.kappa)));
  }
  __syncthreads();
  if (threadIdx.x < 3) d.rowbuf[threadIdx.x * R + J] = seq_acc(row + threadIdx.x * ni, ni) / ni;
}
__global__ void __launch_bounds__(256) k_gzu_core(const MemberDesc *D, int mb) {
  MEMBER;
  if (!d.is_gas) return;
  extern __shared__ double sh[];
  const int nj = d.nj, ni = d.ni, R = nj + 3, NJ = 2 * (nj + 1) + 1;
  double *u1 = sh, *p1 = sh + R, *r1 = sh + 2 * R, *pvr = sh + 3 * R, *pvh = sh + 4 * R, *bern = sh + 5 * R;
  double *kn = sh + 6 * R;
  // the metric columns the serial integral reads, staged once
  double *f = sh + 7 * R, *m = f + NJ, *n = m + NJ, *mn = n + NJ, *mni = mn + NJ;
  for (int J = threadIdx.x; J <= nj; J += blockDim.x) {
    u1[J] = d.rowbuf[J];
    p1[J] = d.rowbuf[R + J];
    r1[J] = d.rowbuf[2 * R + J];
  }
  for (int jj = threadIdx.x; jj < NJ; jj += blockDim.x) {
    f[jj] = d.f[jj];
    m[jj] = d.m[jj];
    n[jj] = d.n[jj];
    mn[jj] = d.mn[jj];
    mni[jj] = d.mn_inv[jj];
  }
  __syncthreads();
  // absolute vorticity of the uniform row field
  for (int J = 1 + threadIdx.x; J <= nj; J += blockDim.x) {
    double f2j = f[2 * J], m2j = m[2 * J], n2j = n[2 * J];
    double mm1i = 1. / m[2 * J - 1], mp1i = 1. / m[2 * J + 1];
    double ze = m2j * ((0. - 0.) + n2j * (u1[J - 1] * mm1i - u1[J] * mp1i));
    pvr[J] = (ze + f2j);
  }
  if (threadIdx.x == 0) {
    double ze = 0.;
    for (int I = 1; I <= ni; I++) ze -= u1[0];
    ze *= mn[0] / ((m[1]) * (double)(ni));
    pvr[0] = ze + f[0];
  } else if (threadIdx.x == 64) {
    double ze = 0.;
    for (int I = 1; I <= ni; I++) ze += u1[nj];
    ze *= mn[2 * (nj + 1)] / (m[2 * nj + 1] * (double)(ni));
    pvr[nj + 1] = ze + f[2 * (nj + 1)];
  }
  __syncthreads();
  for (int J = threadIdx.x; J <= nj + 1; J += blockDim.x) {
    double v = 0.;
    if (J >= 1 && J <= nj) {
      double udyJ = u1[J] / n[2 * J + 1], udyM = u1[J - 1] / n[2 * J - 1];
      // the uniform rows' PV in the weights of the v grid
      auto P = [&](int j, int) { return pvr[j]; };
      const PvW<double> w = pv_weights_v<double>(d.pv_al81, P, J, 1);
      v = (w.ga * udyJ + w.de * udyJ + w.al * udyM + w.be * udyM) * w.coef;
      v += (p1[J] - p1[J - 1]) * 2. / (r1[J] + r1[J - 1]);
    }
    pvh[J] = v;
    if (J <= nj) kn[J] = kin_uniform(mn, mni, nj, u1, J, d.pv_al81);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // Bernoulli function integrated from the tie-point row both ways
    // (running values in a register, in the same order; the increments are
    // read eight at a time ahead of the chain)
    const int j0 = d.jtp;
    const double b0 = 0. + kn[j0];
    bern[j0] = b0;
    double b = b0;
    int J = j0 + 1;
    for (; J + 7 <= nj; J += 8) {
      double q[8];
#pragma unroll
      for (int u = 0; u < 8; u++) q[u] = pvh[J + u];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        b = b - q[u];
        bern[J + u] = b;
      }
    }
    for (; J <= nj; J++) {
      b = b - pvh[J];
      bern[J] = b;
    }
    b = b0;
    J = j0 - 1;
    for (; J - 7 >= 0; J -= 8) {
      double q[8];
#pragma unroll
      for (int u = 0; u < 8; u++) q[u] = pvh[J - u + 1];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        b = b + q[u];
        bern[J - u] = b;
      }
    }
    for (; J >= 0; J--) {
      b = b + pvh[J + 1];
      bern[J] = b;
    }
  }
  __syncthreads();
  for (int J = threadIdx.x; J <= nj + 1; J += blockDim.x) {
    d.rowbuf[3 * R + J] = pvr[J];
    if (J <= nj) d.rowbuf[4 * R + J] = bern[J] - kn[J];
  }
}
void L_gz_from_u(hipStream_t s, const Bucket &b) {
  if (!b.any_gas) return;
  if (b.mixed) LAUNCH_AS("k_gzu_means", k_gzu_means<true>, dim3(b.nj + 1, 1, b.nm), dim3(64), sizeof(double) * 3 * b.ni, s, b.D, b.mb);
  else LAUNCH_AS("k_gzu_means", k_gzu_means<false>, dim3(b.nj + 1, 1, b.nm), dim3(64), sizeof(double) * 3 * b.ni, s, b.D, b.mb);
  LAUNCH(k_gzu_core, dim3(1, 1, b.nm), dim3(256), sizeof(double) * (7 * (b.nj + 3) + 5 * (2 * b.nj + 3)), s, b.D,
         b.mb);
  // GZ_SURFACE and PV3's plane nk+1 are filled in by the k_gz3 that follows
}

// hydrostatic GZ3 and MONT3 from the bottom up (Leslie-Purser 4-point
// integral in ln p) and the monotonicity screen
// FP64, 1024x512x64: 650 us before, 415 now; 256x128x20: 20 and 15.
template <bool F, int KC, bool U>
__global__ void __launch_bounds__(1024) k_gz3(const MemberDesc *D, int mb, int C) {
  MEMBER;
  extern __shared__ double lds[];
  const Tile<U> T(d, C, KC);
  const int nk = d.nk, J = T.J, I = T.I, K0 = T.K0;
  double *L = lds + T.c;  // [K C]: the increment of layer K, then GZ3
  // the column's surface geopotential, read ahead by the lane that runs the
  // chain; on a gas giant gz_from_u's results for this column: GZ_SURFACE,
  // and plane nk+1 of PV3 (the absolute vorticity of the uniform rows; row
  // nj+1 by the columns of row nj)
  double gs = 0.;
  if (T.live && T.scan) {
    if (d.is_gas) {
      const int R = d.nj + 3;
      gs = d.rowbuf[4 * R + J];
      d.GZS[T.i] = gs;
      double *pv = d.PV3 + (size_t)(d.nk + 1) * d.N2;
      pv[T.i] = d.rowbuf[3 * R + J];
      if (J == d.nj) pv[ix2(d, J + 1, I)] = d.rowbuf[3 * R + J + 1];
    } else {
      gs = d.GZS[T.i];
    }
  }
  // P3 and RHO3 on K0-2 .. K0+KC
  double p[KC + 3], rho[KC + 3];
#pragma unroll
  for (int r = 0; r < KC + 3; r++) {
    const int K = min(max(K0 - 2 + r, 0), nk);
    p[r] = T.at(d, d.P3, K)[T.i];
    rho[r] = T.at(d, d.RHO3, K)[T.i];
  }
  // log(P3(K)/P3(K-1)) and P3/RHO3, each once per level of the chunk
  double lg[KC + 2], df[KC + 3];
  m_log2<F>(p[1] / p[0], p[2] / p[1], &lg[0], &lg[1]);
#pragma unroll
  for (int r = 0; r < 3; r++) df[r] = p[r] / rho[r];
#pragma unroll
  for (int r = 0; r < KC; r++) {
    const int K = K0 + r;
    if (r % 2 == 0) m_log2<F>(p[r + 3] / p[r + 2], p[min(r + 4, KC + 2)] / p[r + 3], &lg[r + 2], &lg[min(r + 3, KC + 1)]);
    df[r + 3] = p[r + 3] / rho[r + 3];
    double v;
    if (K >= nk || K == 1) {
      v = ((p[r + 2] + p[r + 1]) / (rho[r + 2] + rho[r + 1])) * lg[r + 1];
    } else {
      const double dz10 = lg[r + 2], dz21 = lg[r + 1], dz32 = lg[r];
      const double dz20 = dz21 + dz10, dz30 = dz32 + dz20, dz31 = dz32 + dz21;
      const double df0 = df[r + 3], df1 = df[r + 2], df2 = df[r + 1], df3 = df[r];
      v = -(df0 * (dz21 * dz21 * dz21 * (dz31 + dz32)) / (dz10 * dz20 * dz30) +
            df1 * (dz21 * (dz21 * (dz21 + 2. * (dz10 - dz31)) - 6. * dz10 * dz31)) / (dz10 * dz31) +
            df2 * (dz21 * (dz21 * (dz21 + 2. * (dz32 - dz20)) - 6. * dz20 * dz32)) / (dz20 * dz32) +
            df3 * (dz21 * dz21 * dz21 * (dz10 + dz20)) / (dz30 * dz31 * dz32)) /
          12.;
    }
    if (K <= nk) L[K * C] = v;
  }
  double t[KC];
#pragma unroll
  for (int r = 0; r < KC; r++) t[r] = T.at(d, d.T3, min(K0 + r, nk))[T.i];
  __syncthreads();
  if (T.scan) {
    double gp = d.topo_scale * gs;
    const bool inner = T.live && (I >= 1 && I <= d.ni);
    int bad = 0;
    // the increments are read eight levels at a time ahead of the chain
    int K = nk;
    for (; K - 7 >= 1; K -= 8) {
      double i8[8];
#pragma unroll
      for (int u = 0; u < 8; u++) i8[u] = L[(K - u) * C];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const double gn = gp + i8[u];
        L[(K - u) * C] = gp;
        if (inner && gp >= gn) bad = 1;
        gp = gn;
      }
    }
    for (; K >= 1; K--) {
      const double gn = gp + L[K * C];
      L[K * C] = gp;
      if (inner && gp >= gn) bad = 1;
      gp = gn;
    }
    L[0] = gp;
    if (bad) atomicOr(&d.dyn->err, 1);
  }
  __syncthreads();
  if (!T.live) return;
  const double cpr = d.cpr, rgas = d.rgas;
  auto out = [&](int K, double tk) {
    const double gz = L[K * C];
    Plane<double>{d.GZ3 + (size_t)K * d.N2}[T.i] = gz;
    Plane<double>{d.MONT3 + (size_t)K * d.N2}[T.i] = gz + cpr * tk * rgas;
  };
  if (T.scan) out(0, T.at(d, d.T3, 0)[T.i]);
#pragma unroll
  for (int r = 0; r < KC; r++) {
    const int K = K0 + r;
    if (K > nk) break;
    out(K, t[r]);
  }
}
template <bool F>
static void gz3_t(hipStream_t s, const Bucket &b) {
  const ColShape sh = col_shape(b, b.knob[KN_COLS_GZ3]);
#define K_(KC, U) k_gz3<F, KC, U>
  COLS_LAUNCH("k_gz3", K_, sh, tile_grid(b, sh.C), dim3(sh.nt), col_lds(b, sh.C), s, b.D, b.mb, sh.C);
#undef K_
}
void L_gz3(hipStream_t s, const Bucket &b) {
  if (b.mixed) gz3_t<true>(s, b);
  else gz3_t<false>(s, b);
}

// finish DZDT3 (diagnostic vertical velocity); in the step k_ab does it where
// it can
__global__ void __launch_bounds__(256) k_dzdt3(const MemberDesc *D, int mb) {
  MEMBER_X;
  FLAT2_X(0, d.nj + 1, 1, d.ni);
  dzdt3_at(d, 1 + bx_.y, J, I);
}
void L_dzdt3(hipStream_t s, const Bucket &b) {
  LAUNCH(k_dzdt3, grid2(b.nj + 1, b.ni, b.nk, b.nm), dim3(TPB), 0, s, b.D, b.mb);
}

// ------------------------------------------------------------ heating
// the Held-Suarez relaxation of a cell from its p, T, the column's bottom
// pressure and (p/p0)^kappa, p0 = 1000 hPa
template <bool F>
__device__ __forceinline__ double hs_relax(const MemberDesc &d, int J, double p, double t, double pbot, double pk0) {
  const double ka = 1. / (40. * 60. * 60. * 24.), ks = 1. / (4. * 60. * 60. * 24.);
  const double dt_y = 60., dth_z = 10., p0 = 1000. * 100.;
  double kt = ka;
  double amp = (p / pbot - 0.7) / (1. - 0.7);
  // cos(lat) and its fourth power from the host tables (the host libm, as
  // the oracle forms them)
  if (amp > 0.) kt += (ks - ka) * d.coslat4_h[J] * amp;
  double t_cool = 1. / kt;
  double cpt = 1004. / t_cool;
  double c2 = d.coslat_h[J];
  c2 *= c2;
  double s2 = 1. - c2, pp0 = p / p0;
  double teq = (315. - dt_y * s2 - dth_z * m_log<F>(pp0) * c2) * pk0;
  teq = dmax(200., teq);
  return -cpt * (t - teq);
}
__device__ double hs_newton(const MemberDesc &d, int K, int J, int I) {
  const double p = d.P3[ix3(d, K, J, I)];
  return hs_relax(d, J, p, d.T3[ix3(d, K, J, I)], d.P3[ix3(d, d.nk, J, I)], crm_pow(p / (1000. * 100.), d.kappa));
}

// Day-night relaxation of the hot-Jupiter case (no reference counterpart):
// HEAT3 = cp (T_eq - T)/tau_rad, T_eq = T_ref(p) + dT(p) (max(0, cos(lat)
// cos(lon)) - 1/4), T_ref the initial profile's temperature, dT the full
// contrast above teq_p_contrast and linear in ln p to 0 at pbot.
// the day-night relaxation of a cell from its p, T, (p/press0)^kappa and the
// column I whose longitude it takes
template <bool F>
__device__ __forceinline__ double hj_relax(const MemberDesc &d, int J, int I, double p, double t, double pk) {
  const double tref = (1. / (1. / d.ref_theta_b + d.ref_a_over_kappa * (pk - d.ref_pbk))) * pk;
  double dT = d.teq_contrast;
  // the per-member log and the per-row/column cosines come from host tables
  // formed with the host libm, as the oracle forms them
  if (p > d.teq_p_contrast) dT *= dmax(0., m_log<F>(d.pbot / p) / d.hj_lnref);
  const double cl = d.coslat_h[J];
  const double day = dmax(0., cl * d.coslon_h[I]);
  const double teq = tref + dT * (day - .25);
  return d.cp * (teq - t) / d.tau_rad;
}
__device__ double hj_newton(const MemberDesc &d, int K, int J, int I) {
  const double p = d.P3[ix3(d, K, J, I)];
  return hj_relax(d, J, I, p, d.T3[ix3(d, K, J, I)], crm_pow(p / d.press0, d.kappa));
}

// HEAT3 = 0 everywhere, then the Held-Suarez, day-night or sounding
// relaxation on K = 1..nk with its zonal pads (the bc_lateral at the end of
// calc_heating)
__global__ void __launch_bounds__(256) k_heating(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 1, d.ni);
  const int K = 1 + blockIdx.y;
  if (!newt_relax_on(d)) return;
  double h;
  if (d.is_tab) {
    const size_t q = ix3(d, K, J, I);
    h = 0. + tab_relax(d, d.P3[q], d.T3[q]);
  } else {
    h = d.is_hj ? hj_newton(d, K, J, I) : 0. + hs_newton(d, K, J, I);
  }
  d.HEAT3[ix3(d, K, J, I)] = h;
  if (I == d.ni) d.HEAT3[ix3(d, K, J, 0)] = h;
  if (I == 1) d.HEAT3[ix3(d, K, J, d.ni + 1)] = h;
}
// Layer-mean removal of the relaxation (K <= k_sponge or newt_cool_adjust,
// src/shared/epic_sensible_heating.c:139-167), from the relaxation HEAT3
// holds: one block per layer stages rows of HEAT3 times the cell area
// 1/mn in LDS, and one lane adds them in the reference's order (J, then I);
// the total area, which depends on the metric only, is formed on the host
// by the same loop.  The layer mean goes to sD[K].
__global__ void __launch_bounds__(256) k_heat_layer_mean(const MemberDesc *D, int mb) {
  MEMBER;
  extern __shared__ double lds[];
  const int K = 1 + blockIdx.x;
  if (!newt_relax_on(d)) return;
  if (!(K <= d.k_sponge || d.newt_cool_adjust)) return;
  const int ni = d.ni, nrow = d.nj + 1;
  const int rpc = (2048 / ni) > 0 ? 2048 / ni : 1;  // rows per LDS chunk
  double ha = 0.;
  for (int j0 = 0; j0 < nrow; j0 += rpc) {
    const int nr = (nrow - j0) < rpc ? (nrow - j0) : rpc;
    for (int t = threadIdx.x; t < nr * ni; t += blockDim.x) {
      const int J = j0 + t / ni, I = 1 + t % ni;
      const double da = 1. / d.mn[2 * J + 1];
      lds[t] = d.HEAT3[ix3(d, K, J, I)] * da;
    }
    __syncthreads();
    if (threadIdx.x == 0) ha = seq_acc(lds, nr * ni, ha);
    __syncthreads();
  }
  if (threadIdx.x == 0) d.sD[K] = ha / d.heat_area;
}
__global__ void __launch_bounds__(256) k_heat_adjust_apply(const MemberDesc *D, int mb) {
  MEMBER;
  FLAT2(0, d.nj + 1, 0, d.ni + 2);
  const int K = 1 + blockIdx.y;
  if (!newt_relax_on(d)) return;
  if (!(K <= d.k_sponge || d.newt_cool_adjust)) return;
  const size_t q = ix3(d, K, J, I);
  d.HEAT3[q] = 0. + (d.HEAT3[q] - d.sD[K]);
}
// in_thermo: the relaxation was formed by this step's k_thermo,
// and every other cell of HEAT3 is zero (a member's blob is cleared when it
// is created, a drop-in upload brings the caller's array, which the
// reference zeroes there, and no kernel writes outside K = 1..nk, J = 0..nj),
// so only the layer-mean adjustment is left
void L_heating(hipStream_t s, const Bucket &b, int adjust, bool in_thermo) {
  if (!in_thermo) {
    L_fill(s, b, F_HEAT3, 0.);
    LAUNCH(k_heating, grid2(b.nj + 1, b.ni, b.nk, b.nm), dim3(TPB), 0, s, b.D, b.mb);
  }
  if (adjust) {
    LAUNCH(k_heat_layer_mean, dim3(b.nk, 1, b.nm), dim3(256), sizeof(double) * 2048, s, b.D, b.mb);
    LAUNCH(k_heat_adjust_apply, grid2(b.nj + 1, b.ni + 2, b.nk, b.nm), dim3(TPB), 0, s, b.D, b.mb);
  }
}

// ------------------------------------------------------------ calc_w
// Column tiles.  Per level: the theta heating of source_sink
// (src/shared/epic_funcs_diag.c:4768-4778, with_source), the heating part
// of W3, the Leslie-Purser increment of SUM_DIV and dF/dp; then the running
// SUM_DIV in one lane per column.  SUM_DIV(1) and SUM_DIV(nk) are zero (the
// reference's top/bottom statements write stale-index pad cells), so the
// dF/dpbot term vanishes and is not formed.
// With with_source (the step's call) the blocks past the ncb column tiles
// first clear what the step does not write of its tendency planes of u and v
// (the FP64 plane IT_ZERO, or the mixed mode's one FP64 plane; nothing in this
// launch reads them): planes 0, nk and nk+1 and, of the planes between, rows
// -1, 0 and nj+1.  k_uv_core forms the rest (row 0 of u again) and k_filter3
// writes the pads of the rows it passes.
// FP64, 1024x512x64: 1065 us before, 774 now; 256x128x20: 35 both.
template <bool F, int KC, bool U>
__global__ void __launch_bounds__(1024) k_calc_w(const MemberDesc *D, int mb, int with_source, int C, int ncb) {
  MEMBER;
  if ((int)blockIdx.x >= ncb) {
    const size_t off = d.mixed ? 0 : (size_t)d.dyn->it0 * d.N3;
    double *du = d.DUDT + off, *dv = d.DVDT + off;
    const int st = (gridDim.x - ncb) * blockDim.x, n = 3 * d.N2 + 3 * d.Ia * (d.nk - 1);
    for (int i = (blockIdx.x - ncb) * blockDim.x + threadIdx.x; i < n; i += st) {
      size_t q;
      if (i < 3 * d.N2) {
        const int p = i / d.N2;
        q = (size_t)(p == 0 ? 0 : d.nk + p - 1) * d.N2 + (i - p * d.N2);
      } else {
        const int e = i - 3 * d.N2, row = e / d.Ia, k = row / 3, r = row - 3 * k;
        q = ix3(d, 1 + k, r == 0 ? -1 : r == 1 ? 0 : d.nj + 1, e - row * d.Ia);
      }
      du[q] = 0.;
      dv[q] = 0.;
    }
    return;  // a whole block: no barrier below waits for it
  }
  extern __shared__ double lds[];
  const Tile<U> T(d, C, KC);
  const int nk = d.nk, ks = d.ks, K0 = T.K0;
  double *L = lds + T.c;  // [K C]: the increment of SUM_DIV, then SUM_DIV
  int bad = 0;
  const double ptop = T.at(d, d.P3, 0)[T.i], pbot = T.at(d, d.P3, nk)[T.i], psig = T.at(d, d.P3, ks - 1)[T.i];
  // SUM_DIV's increments: P3 and the divergence on K0-2 .. K0+KC, their
  // product and log(P3(K)/P3(K-1)), the ln-p interval of the Leslie-Purser
  // weights, once per level of the chunk
  double p3[KC];
  {
    double p[KC + 3], f[KC + 3], lg[KC + 2];
#pragma unroll
    for (int r = 0; r < KC + 3; r++) {
      const int K = min(max(K0 - 2 + r, 0), nk);
      p[r] = T.at(d, d.P3, K)[T.i];
      f[r] = T.at(d, d.DIV, K)[T.i];
    }
#pragma unroll
    for (int r = 0; r < KC; r++) p3[r] = p[r + 2];
#pragma unroll
    for (int r = 0; r < KC + 3; r++) f[r] = p[r] * f[r];
    m_log2<F>(p[1] / p[0], p[2] / p[1], &lg[0], &lg[1]);
#pragma unroll
    for (int r = 0; r < KC; r++) {
      const int K = K0 + r;
      if (r % 2 == 0) m_log2<F>(p[r + 3] / p[r + 2], p[min(r + 4, KC + 2)] / p[r + 3], &lg[r + 2], &lg[min(r + 3, KC + 1)]);
      double ds = 0.;
      if (K >= 2) {
        const double dz10 = lg[r], dz21 = lg[r + 1], dz32 = lg[r + 2];
        const double dz20 = dz21 + dz10, dz30 = dz32 + dz20, dz31 = dz32 + dz21;
        const double df0 = f[r], df1 = f[r + 1], df2 = f[r + 2], df3 = f[r + 3];
        ds = -(df0 * (dz21 * dz21 * dz21 * (dz31 + dz32)) / (dz10 * dz20 * dz30) +
               df1 * (dz21 * (dz21 * (dz21 + 2. * (dz10 - dz31)) - 6. * dz10 * dz31)) / (dz10 * dz31) +
               df2 * (dz21 * (dz21 * (dz21 + 2. * (dz32 - dz20)) - 6. * dz20 * dz32)) / (dz20 * dz32) +
               df3 * (dz21 * dz21 * dz21 * (dz10 + dz20)) / (dz30 * dz31 * dz32)) /
             12.;
      }
      if (K < nk) L[K * C] = ds;
    }
  }
  __syncthreads();
  if (T.scan) {
    // (read eight levels at a time ahead of the chain)
    double S = 0.;
    int K = 2;
    for (; K + 7 < nk; K += 8) {
      double s8[8];
#pragma unroll
      for (int u = 0; u < 8; u++) s8[u] = L[(K + u) * C];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        S = S + s8[u];
        L[(K + u) * C] = S;
      }
    }
    for (; K < nk; K++) {
      S = S + L[K * C];
      L[K * C] = S;
    }
  }
  __syncthreads();
  // theta with its heating, the heating's part of W3 and dF/dp
  const double eps = d.eps13, lr = m_log<F>(ptop / pbot);
  auto out = [&](double *f, int K, double x) {
    if (T.live) Plane<double>{f + (size_t)K * d.N2}[T.i] = x;
  };
  if (T.scan) out(d.W3, 0, 0.);
  constexpr int KB = 2;  // levels loaded together
#pragma unroll
  for (int rb = 0; rb < KC; rb += KB) {
    double th[KB], heat[KB], ex[KB];
#pragma unroll
    for (int r = 0; r < KB; r++) {
      const int K = min(K0 + rb + r, nk);
      th[r] = T.at(d, d.THETA, K)[T.i];
      heat[r] = T.at(d, d.HEAT3, K)[T.i];
      ex[r] = T.at(d, d.EXNER3, K)[T.i];
    }
#pragma unroll
    for (int r = 0; r < KB; r++) {
      const int K = K0 + rb + r;
      if (K > nk) break;
      const double pc = p3[rb + r];
      if (with_source && K >= ks - 1) {
        th[r] += d.dt * heat[r] / ex[r];
        out(d.THETA, K, th[r]);
      }
      if (K == nk) {
        out(d.W3, nk, 0.);
        break;
      }
      double wb = 0.;
      if (K < ks - 1) wb = g_sig<F>(d, get_sigma_l<F>(pbot, pc, lr)) * heat[r] / ex[r];
      const double dp = pc * eps;
      double p2 = dmax(pc - dp * .5, ptop), dF = 0.;
      const double p4 = dmin(pc + dp * .5, pbot);
      if (p2 < psig && p4 >= psig) p2 = pc;
      if (p2 < p4) dF = sgth_diff_l<F>(d, th[r], p2, p4, pbot, ptop, lr, &bad) / (p2 - p4);
      else bad = 1;
      out(d.W3, K, wb - L[K * C] * dF);  // (SUM_DIV(1) is 0, as its L was left)
    }
  }
  if (bad) atomicOr(&d.dyn->err, 2);
}
template <bool F>
static void calc_w_t(hipStream_t s, const Bucket &b, int with_source) {
  const ColShape sh = col_shape(b, b.knob[KN_COLS_CALCW]);
  dim3 g = tile_grid(b, sh.C);
  const int ncb = (int)g.x;
  if (with_source) {
    // blocks that clear the tendencies' edges: about 4 cells per lane
    const size_t n = (size_t)(b.ni + 2) * (3 * (b.nj + 3) + 3 * (b.nk - 1));
    g.x += (unsigned)std::max<size_t>(1, std::min<size_t>(1024, n / ((size_t)sh.nt * 4)));
  }
#define K_(KC, U) k_calc_w<F, KC, U>
  COLS_LAUNCH("k_calc_w", K_, sh, g, dim3(sh.nt), col_lds(b, sh.C), s, b.D, b.mb, with_source, sh.C, ncb);
#undef K_
}
void L_calc_w(hipStream_t s, const Bucket &b, int with_source) {
  if (b.mixed) calc_w_t<true>(s, b, with_source);
  else calc_w_t<false>(s, b, with_source);
}

// ------------------------------------------------ vorticity / divergence
// PV3 planes k0..k1 from U (uu) and the zonally filtered V (vv), with H3.
// One block per (K,J) pv-row group: row J of vv is filtered by its lanes
// (rows of the v-grid filter band), which hand each other their neighbours
// through the row's ni values of LDS.  A lane's four points are written out,
// so their loads are in flight together.  bx is the row group.
template <bool WIDE>
__device__ __forceinline__ void vort_interior_rows(const MemberDesc &d, double *lds, int bx, int K, int uf, int vf) {
  const RowMap m = row_map(d.ni);
  const int Jr = 1 + bx * m.rpb + m.g, ni = d.ni;
  const bool live = Jr <= d.nj;
  const int J = live ? Jr : 1;
  const Plane<const double> uu{fld_ptr(d, uf) + (size_t)K * d.N2}, vv{fld_ptr(d, vf) + (size_t)K * d.N2};
  const Plane<const double> hh{d.H3 + (size_t)K * d.N2};
  const Plane<double> pv{d.PV3 + (size_t)K * d.N2};
  double *xv = lds + (size_t)m.g * ni;  // xv[I-1] = filtered vv(J,I)
  double v[4], u0[4], u1[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    v[q] = vv[ix2(d, J, I)];
    u0[q] = uu[ix2(d, J - 1, I)];
    u1[q] = uu[ix2(d, J, I)];
  }
  const bool filt = live && d.rflag_v[J] != 0;
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, v, xv, J, 1, filt, m.lane);
#pragma unroll
  for (int q = 0; q < 4; q++) xv[m.lane + m.stride * q] = v[q];
  row_sync<WIDE>();
  if (!live) return;
  double f2j = d.f[2 * J], m2j = d.m[2 * J], n2j = d.n[2 * J];
  double mm1i = 1. / d.m[2 * J - 1], mp1i = 1. / d.m[2 * J + 1];
  double mnm1i = 1. / d.mn[2 * J - 1], mnp1i = 1. / d.mn[2 * J + 1];
  double mn_pv = .5 / (mnm1i + mnp1i);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    const double vc = v[q], vw = xv[I == 1 ? ni - 1 : I - 2];
    double ze = m2j * ((vc - vw) + n2j * (u0[q] * mm1i - u1[q] * mp1i));
    double w = (ze + f2j);
    double h_pv = ((hh[ix2(d, J, I)] + hh[ix2(d, J, I - 1)]) * mnp1i +
                   (hh[ix2(d, J - 1, I)] + hh[ix2(d, J - 1, I - 1)]) * mnm1i) * mn_pv;
    w /= h_pv;
    pv[ix2(d, J, I)] = w;
    if (I == ni) pv[ix2(d, J, 0)] = w;
    if (I == 1) pv[ix2(d, J, ni + 1)] = w;
  }
}
// pole PV from the circulation of the adjacent u-row (north = 1: J = nj+1
// from row nj, else J = 0 from row 0): the row is staged in LDS and lanes
// 0/1 form the two zonal sums in the reference's sequential order.  Every
// lane of the block reaches both barriers.
__device__ __forceinline__ void vort_pole(const MemberDesc &d, double *row, int K, int north, int uf) {
  const Plane<const double> uu{fld_ptr(d, uf) + (size_t)K * d.N2};
  const Plane<const double> hh{d.H3 + (size_t)K * d.N2};
  const Plane<double> pv{d.PV3 + (size_t)K * d.N2};
  const int ni = d.ni, nj = d.nj, Jr = north ? nj : 0;
  for (int i = threadIdx.x; i < ni; i += blockDim.x) {
    row[i] = uu[ix2(d, Jr, i + 1)];
    row[ni + i] = hh[ix2(d, Jr, i + 1)];
  }
  __syncthreads();
  double *res = row + 2 * ni;
  if (threadIdx.x == 0) {
    double ze;
    if (!north) {
      ze = seq_acc<true>(row, ni);
      ze *= d.mn[0] / ((d.m[1]) * (double)(ni));
    } else {
      ze = seq_acc(row, ni);
      ze *= d.mn[2 * (nj + 1)] / (d.m[2 * nj + 1] * (double)(ni));
    }
    res[0] = ze;
  } else if (threadIdx.x == 1) {
    double h = seq_acc(row + ni, ni);
    h /= (double)(ni);
    res[1] = h;
  }
  __syncthreads();
  const double val = (res[0] + (north ? d.f[2 * (nj + 1)] : d.f[0])) / res[1];
  const int Jd = north ? nj + 1 : 0;
  for (int I = threadIdx.x; I <= ni + 1; I += blockDim.x) pv[ix2(d, Jd, I)] = val;
}
// DIV of (uu zonally filtered, vv) on plane K: one block per (K,J) h-row
// group, row J of uu filtered by its lanes (rows of the h-grid filter band)
template <bool WIDE>
__device__ __forceinline__ void divergence_rows(const MemberDesc &d, double *lds, int bx, int K, int uf, int vf, int df) {
  const RowMap m = row_map(d.ni);
  const int Jr = bx * m.rpb + m.g, ni = d.ni;
  const bool live = Jr <= d.nj;
  const int J = live ? Jr : 0;
  const Plane<const double> uu{fld_ptr(d, uf) + (size_t)K * d.N2}, vv{fld_ptr(d, vf) + (size_t)K * d.N2};
  const Plane<double> di{fld_ptr(d, df) + (size_t)K * d.N2};
  double *xu = lds + (size_t)m.g * ni;  // xu[I-1] = filtered uu(J,I)
  double u[4], v0[4], v1[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    u[q] = uu[ix2(d, J, I)];
    v0[q] = vv[ix2(d, J, I)];
    v1[q] = vv[ix2(d, J + 1, I)];
  }
  const bool filt = live && d.rflag_h[J] != 0;
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, u, xu, J, 0, filt, m.lane);
#pragma unroll
  for (int q = 0; q < 4; q++) xu[m.lane + m.stride * q] = u[q];
  row_sync<WIDE>();
  if (!live) return;
  int jj = 2 * J + 1;
  double n_inv = 1. / d.n[jj], mn = d.mn[jj];
  double m2j_inv = (J == 0) ? 0. : 1. / d.m[jj - 1];
  double m2jp2_inv = (J == d.nj) ? 0. : 1. / d.m[jj + 1];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    const double ue = xu[I == ni ? 0 : I], uc = u[q];
    double w = mn * ((ue * n_inv - uc * n_inv) + (v1[q] * m2jp2_inv - v0[q] * m2j_inv));
    di[ix2(d, J, I)] = w;
    if (I == ni) di[ix2(d, J, 0)] = w;
    if (I == 1) di[ix2(d, J, ni + 1)] = w;
  }
}

template <bool WIDE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_divergence(const MemberDesc *D, int mb, int uf, int vf, int df, int k0) {
  MEMBER;
  extern __shared__ double lds[];
  divergence_rows<WIDE>(d, lds, blockIdx.x, k0 + blockIdx.y, uf, vf, df);
}

// store_diag in one launch: on planes K = 0..nk, blocks [0, nv) form the PV
// rows, [nv, nv + nd) the divergence rows, and the last two the pole PV of
// the plane (the three are independent: each reads U, V and H3 only).  With
// rotate set, the first block of plane 0 of each member then rotates its
// time planes (IT_ZERO <- IT_MINUS2 <- IT_MINUS1 <- IT_ZERO) and advances
// itime: the step's last use of them was its Adams-Bashforth update, and no
// block of this launch reads them.
template <bool WIDE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_store_diag(const MemberDesc *D, int mb, int nv, int nd, int rotate) {
  MEMBER;
  extern __shared__ double lds[];
  const int bx = blockIdx.x, K = blockIdx.y;
  if (bx < nv) vort_interior_rows<WIDE>(d, lds, bx, K, F_U, F_V);
  else if (bx < nv + nd) divergence_rows<WIDE>(d, lds, bx - nv, K, F_U, F_V, F_DIV);
  else vort_pole(d, lds, K, bx - nv - nd, F_U);
  if (rotate && bx == 0 && K == 0 && threadIdx.x == 0) {
    MemberDyn *y = d.dyn;
    int t = y->itm2;
    y->itm2 = y->itm1;
    y->itm1 = y->it0;
    y->it0 = t;
    y->itime += 1;
  }
}
void L_store_diag(hipStream_t s, const Bucket &b, int rotate) {
  const int rpb = rows_per_block(b.ni);
  const int nv = (b.nj + rpb - 1) / rpb, nd = (b.nj + 1 + rpb - 1) / rpb;
  const size_t shm = sizeof(double) * std::max(rpb * b.ni, 2 * b.ni + 2);
  ROWS_LAUNCH(b, "k_store_diag", k_store_diag<true>, k_store_diag<false>, dim3(nv + nd + 2, b.nk + 1, b.nm), dim3(256), shm, s, b.D, b.mb, nv, nd, rotate);
}
void L_divergence(hipStream_t s, const Bucket &b, int uu, int vv, int dst, int k0, int k1) {
  const int rpb = rows_per_block(b.ni);
  ROWS_LAUNCH(b, "k_divergence", k_divergence<true>, k_divergence<false>, dim3((b.nj + 1 + rpb - 1) / rpb, k1 - k0 + 1, b.nm), dim3(256), sizeof(double) * rpb * b.ni, s,
         b.D, b.mb, uu, vv, dst, k0);
}

}  // namespace epic
