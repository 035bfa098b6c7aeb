// k_adv.hip -- flux-form predictor-corrector advection of Hsu & Arakawa as
// modified by Konor & Arakawa (hsu_advection, src/shared/epic_flux.c:652-1488),
// the monotonized fourth-order centred scheme offered beside it (Akima,
// akima_advection, src/shared/epic_flux.c:1502-1924), and their driver
// (advection, src/shared/epic_flux.c:346-637).
//
// Directions are split as in the reference: vertical column pass, then a
// meridional pass on every level, then a zonal pass on a zonally filtered
// copy.  The column pass works on LDS column tiles, the meridional pass on
// LDS tiles of a few rows by up to 64 columns (each intermediate of the
// tile formed once), the zonal pass on LDS rows; every intermediate value
// is formed by the same expression as in the reference, so nothing changes
// but where it is computed.
//
// The three advected fields (unity on the pressure grid, theta, hdry) are
// independent of one another until the theta correction that follows them,
// so every launch of the column and meridional passes carries all three:
// blockIdx.z = field * members + member, each field with its own scratch
// copy (sA + field * N3).
//
// The passes run out of place, field -> adv_out -> sA -> field, so that no
// copy of a field is made: the column pass reads the field (unity is the
// constant 1 and is not read at all; hdry is read with the restore_mass that
// precedes the advection) and leaves its result in adv_out; the meridional
// pass leaves its in sA; the zonal pass filters its row in place of a copy
// of the field and writes the field, theta with its correction (the theta of
// before the passes is still in place then, and the same block has advected
// unity) and hdry with the restore_mass that follows.  Of unity only the
// levels whose correction is used, K >= k_sigma-1, are advected.
//
// The reference keeps its column work arrays in statics across calls: the
// theta call starts at K = k_sigma-1 and reads wm[k_sigma-2] and
// w_a[k_sigma-3] as left by the last column (J = nj, I = ni+1) of the
// preceding unity call.  Both are functions of W3 and of unity before its
// advection (1 everywhere), so the theta blocks form them themselves.
#include "kernels.h"
#include "filter_row.h"

namespace epic {

#define MEMBER const MemberDesc &d = D[mb + blockIdx.z]
// field and member of a block; so: offset of the field's scratch copies
#define ADV_MEMBER                                          \
  const int which = (int)blockIdx.z / nm;                   \
  const MemberDesc &d = D[mb + (int)blockIdx.z - which * nm]; \
  const size_t so = (size_t)which * d.N3
constexpr int ADV_FIELDS = 3;

enum { AV_P3 = 0, AV_THETA = 1, AV_HDRY = 2 };

// where the column pass leaves its result
__device__ __forceinline__ double *adv_out(const MemberDesc &d, int which) {
  return which == AV_P3 ? d.vunity : (which == AV_THETA ? d.vtheta : d.sC);
}
// the field as it enters the advection: hv set, the hyperviscosity left theta
// and hdry in sD's copies 2 and 1 (k_hv4)
__device__ __forceinline__ const double *adv_in(const MemberDesc &d, int which, int hv) {
  if (hv) return d.sD + (size_t)(which == AV_THETA ? 2 : 1) * d.N3;
  return which == AV_THETA ? d.THETA : d.HDRY;
}
// its value on level K at offset q as the column pass takes it (theta above
// its first advected level, which the pass reads too, is the field's)
__device__ __forceinline__ double adv_value(const MemberDesc &d, int which, int K, size_t q, int hv) {
  if (which == AV_P3) return 1.;
  if (which == AV_THETA) return adv_in(d, which, hv && K >= d.ks - 1)[q];
  return dmax(d.h_min[K], adv_in(d, which, hv)[q]);
}
// first level of a field that is advected
__device__ __forceinline__ int adv_kfirst(const MemberDesc &d, int which) { return which == AV_HDRY ? 1 : d.ks - 1; }

// ------------------------------------------------------------ vertical
// Column tiles of C columns (J = 0..nj, I = 1..ni) with every level in LDS.
// The pass is a chain of K-stencils (first-guess flux, predictor, centred
// flux, limiter correction, update) with no recurrence, so each stage runs
// on all lanes over (column, level) pairs, separated by barriers.
//
// The advection passes are templated on the arithmetic type T of the fluxes:
// double reproduces the reference operation for operation; float is the
// mixed mode's (the fields stay FP64: each update adds the FP32 flux
// divergence to the FP64 value).
template <class T> __device__ __forceinline__ T tmin(T x, T y) { return x < y ? x : y; }
template <class T> __device__ __forceinline__ T tmax(T x, T y) { return x > y ? x : y; }

template <class T>
__device__ __forceinline__ T tt_layer(const T *wa, int K, int nk, T ep) {
  T tt;
  if (K == 1) tt = fabs(wa[K + 1] - wa[K]) + ep;
  else if (K == nk) tt = fabs(-wa[K] + wa[K - 1]) + ep;
  else tt = fabs(wa[K + 1] - T(2.) * wa[K] + wa[K - 1]) + ep;
  return tt * tt;
}
template <class T>
__device__ __forceinline__ T tt_iface(const T *wa, int K, int nk, T ep) {
  T tt;
  if (K == 0) tt = fabs(wa[K + 1] - wa[K]) + ep;
  else if (K == nk) tt = fabs(-wa[K] + wa[K - 1]) + ep;
  else tt = fabs(wa[K + 1] - T(2.) * wa[K] + wa[K - 1]) + ep;
  return tt * tt;
}

// The FP64 value a pass updates: the staged copy itself when the pass
// computes in FP64 (the same bits), else a re-read of the FP64 field
__device__ __forceinline__ double old_value(double staged, const double *) { return staged; }
__device__ __forceinline__ double old_value(float, const double *p) { return *p; }
__device__ __forceinline__ double col_value(double staged, const MemberDesc &, int, int, size_t, int) { return staged; }
__device__ __forceinline__ double col_value(float, const MemberDesc &d, int which, int K, size_t q, int hv) {
  return adv_value(d, which, K, q, hv);
}

template <class T>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) k_hsu_vert(const MemberDesc *D, int mb, int nm, int C, int hv) {
  ADV_MEMBER;
  if (d.adv_akima[which]) return;  // the field takes the Akima scheme (uniform per block)
  extern __shared__ double lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);
  const int c = threadIdx.x % C, kk = threadIdx.x / C, KS = blockDim.x / C;
  const int col = blockIdx.x * C + c;
  const bool live = col < (d.nj + 1) * d.ni;
  const int J = live ? col >> d.nlogn : 0, I = live ? 1 + (col & (d.ni - 1)) : 1;
  const int nk = d.nk, L = nk + 2;
  const int layer = (which == AV_HDRY);
  const int kf = (which == AV_THETA) ? d.ks - 1 : 1;
  const T ep = T(1.e-10), DT = T(d.dt);
  const double *dsi = d.dsgth_inv;
  double *out = adv_out(d, which);
  T *wa = lds + c * L, *wv = lds + (C + c) * L, *pr = lds + (2 * C + c) * L, *ff = lds + (3 * C + c) * L;
  // stage 1: field and vertical velocity (wv holds w on the points the
  // field lives on: W3 itself for layers, the interface average otherwise)
  if (live) {
    for (int K = kk; K <= nk + 1; K += KS) {
      double x = 0., w = 0.;
      if (layer) {
        if (K >= kf && K <= nk) x = adv_value(d, which, K, ix3(d, K, J, I), hv);
        if (K >= kf - 1 && K <= nk) w = d.W3[ix3(d, K, J, I)];
      } else {
        if (K >= kf - 1 && K <= nk) x = adv_value(d, which, K, ix3(d, K, J, I), hv);
        if (K >= kf && K <= nk) w = (K == 1 || K == nk) ? 0. : .5 * (d.W3[ix3(d, K, J, I)] + d.W3[ix3(d, K - 1, J, I)]);
        // statics left by the unity pass (wm[kf-1], wa[kf-2] of its last column)
        if (which == AV_THETA && K == kf - 1 && K >= 1) {
          const int Jl = d.nj, Il = d.ni + 1;
          w = dmin(0., (K == 1 || K == nk) ? 0. : .5 * (d.W3[ix3(d, K, Jl, Il)] + d.W3[ix3(d, K - 1, Jl, Il)]));
        }
        if (which == AV_THETA && K == kf - 2) x = 1.;
      }
      wa[K] = T(x);
      wv[K] = T(w);
    }
  }
  __syncthreads();
#define WM(k) tmin(T(0.), wv[k])
#define WP(k) tmax(T(0.), wv[k])
  if (layer) {
    // first-guess flux on interfaces kf..nk-1 (zero at kf-1 and nk)
    if (live)
      for (int K = kf - 1 + kk; K <= nk; K += KS)
        ff[K] = (K == kf - 1 || K == nk) ? T(0.) : WP(K) * wa[K + 1] + WM(K) * wa[K];
    __syncthreads();
    if (live)
      for (int K = kf + kk; K <= nk; K += KS) pr[K] = wa[K] + (ff[K] - ff[K - 1]) * T(dsi[2 * K]) * DT;
    __syncthreads();
    if (live)
      for (int K = kf + kk; K < nk; K += KS)
        ff[K] = T(.5) * (WP(K) * (pr[K] + wa[K + 1]) + WM(K) * (pr[K + 1] + wa[K]));
    __syncthreads();
    if (live)
      for (int K = kf + kk; K < nk; K += KS) {
        const T d1K = pr[K] - wa[K + 1];
        const T d1P = (K + 1 == nk) ? T(0.) : pr[K + 1] - wa[K + 2];
        const T d2K = (K == 1) ? T(0.) : pr[K] - wa[K - 1];
        const T d2P = pr[K + 1] - wa[K];
        const T aaK = tt_layer(wa, K, nk, ep), aaP = tt_layer(wa, K + 1, nk, ep);
        const T aminK = (K >= kf) ? T(d.h_min[K]) : T(0.), aminP = T(d.h_min[K + 1]);
        const T wpK = WP(K), wmK = WM(K);
        T whp = sqrt(wpK * WP(K + 1)), whm = -sqrt(wmK * WM(K - 1));
        T mu = (wpK - wmK) * T(dsi[2 * K + 1]) * DT, al = (T(1.) + mu) / T(6.);
        T gp = aaP / (aaP + (wa[K + 1] - aminP) * (wa[K] - aminK));
        gp = gp * gp;
        T gm = aaK / (aaK + (wa[K + 1] - aminP) * (wa[K] - aminK));
        gm = gm * gm;
        T bp = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gp, bm = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gm;
        T bhp = T(1.) - gp, bhm = T(1.) - gm;
        ff[K] += -al * (wpK * bp * d1K - whp * bhp * d1P + wmK * bm * d2P - whm * bhm * d2K);
      }
    __syncthreads();
    if (live)
      for (int K = kf + kk; K <= nk; K += KS)
        out[ix3(d, K, J, I)] =
            col_value(wa[K], d, which, K, ix3(d, K, J, I), hv) + (double)((ff[K] - ff[K - 1]) * T(dsi[2 * K]) * DT);
  } else {
    // unity's levels above k_sigma-1 serve their neighbours only: flux and
    // predictor from k_sigma-2, the corrected flux from k_sigma-1
    const int k1 = max(kf, d.ks - 2), k2 = max(kf, d.ks - 1);
    // first-guess flux on layers kf..nk (zero below the bottom)
    if (live)
      for (int K = k1 + kk; K <= nk + 1; K += KS) ff[K] = (K == nk + 1) ? T(0.) : WP(K) * wa[K] + WM(K) * wa[K - 1];
    __syncthreads();
    if (live)
      for (int K = max(kf - 1, d.ks - 2) + kk; K <= nk; K += KS)
        pr[K] = (K == kf - 1) ? wa[K] : wa[K] + (ff[K + 1] - ff[K]) * T(dsi[2 * K + 1]) * DT;
    __syncthreads();
    if (live)
      for (int K = k2 + kk; K <= nk; K += KS)
        ff[K] = T(.5) * (WP(K) * (pr[K - 1] + wa[K]) + WM(K) * (pr[K] + wa[K - 1]));
    __syncthreads();
    if (live)
      for (int K = k2 + kk; K <= nk; K += KS) {
        const T d1K = pr[K - 1] - wa[K];
        const T d2K = pr[K] - wa[K - 1];
        const T d2M = (K == kf) ? T(0.) : pr[K - 1] - wa[K - 2];
        const T aaK = tt_iface(wa, K, nk, ep), aaM = tt_iface(wa, K - 1, nk, ep);
        const T wpK = WP(K), wmK = WM(K);
        T whm = (K == 1) ? T(0.) : -sqrt(wmK * WM(K - 1));
        T whp = (K == nk) ? T(0.) : sqrt(wpK * WP(K + 1));
        T mu = (wpK - wmK) * T(dsi[2 * K]) * DT, al = (T(1.) + mu) / T(6.);
        T gp = aaK / (aaK + (wa[K] - T(0.)) * (wa[K - 1] - T(0.)));
        gp = gp * gp;
        T gm = aaM / (aaM + (wa[K] - T(0.)) * (wa[K - 1] - T(0.)));
        gm = gm * gm;
        T bp = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gp, bm = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gm;
        T bhp = T(1.) - gp, bhm = T(1.) - gm, g;
        if (K < nk) {
          const T d1P = pr[K] - wa[K + 1];
          g = -al * (wpK * bp * d1K - whp * bhp * d1P + wmK * bm * d2K - whm * bhm * d2M);
        } else {
          g = -al * (wpK * bp * d1K + wmK * bm * d2K - whm * bhm * d2M);
        }
        ff[K] += g;
      }
    __syncthreads();
    if (live)
      for (int K = k2 + kk; K <= nk; K += KS)
        out[ix3(d, K, J, I)] =
            col_value(wa[K], d, which, K, ix3(d, K, J, I), hv) + (double)((ff[K + 1] - ff[K]) * T(dsi[2 * K + 1]) * DT);
  }
#undef WM
#undef WP
}

// ---------------------------------------------------------- meridional
// One launch: a block holds a tile of TJ rows x CW columns of one plane of
// one field in LDS, with halos: the field on rows J0-2..J0+TJ+1, the
// meridional velocities vp, vm (v times 1/m, split by sign) on v-rows
// J0-1..J0+TJ+1, the smoothness terms aq and the predictor ap on rows
// J0-1..J0+TJ and the corrected flux on v-rows J0..J0+TJ, each formed once per
// cell by the reference's expression (the halo rows are formed again by the
// neighbouring tile: the same values).  The update goes to sA.
template <class T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_hsu_mer(const MemberDesc *D, int mb, int nm, int CW, int MER_TJ) {
  ADV_MEMBER;
  const int K = 1 + blockIdx.y;
  if (d.adv_akima[which] || K < adv_kfirst(d, which)) return;  // uniform per block
  extern __shared__ double sh_raw[];
  T *sh = reinterpret_cast<T *>(sh_raw);
  const int nj = d.nj, nchunk = d.ni / CW;
  const int tile = blockIdx.x / nchunk, chunk = blockIdx.x - tile * nchunk;
  const int J0 = tile * MER_TJ, c = threadIdx.x % CW, r0 = threadIdx.x / CW, RS = blockDim.x / CW;
  const int I = 1 + chunk * CW + c;
  const int RA = MER_TJ + 4, RV = MER_TJ + 3, RP = MER_TJ + 2;
  T *ta = sh, *tvp = ta + RA * CW, *tvm = tvp + RV * CW, *taq = tvm + RV * CW, *tap = taq + RP * CW;
  T *tff = tap + RP * CW;
  const size_t o = (size_t)K * d.N2;
  const Plane<const double> A{adv_out(d, which) + o};
  const T amin = (which == AV_HDRY) ? T(d.h_min[K]) : T(0.), DT = T(d.dt), ep = T(1.e-10);
  // row index helpers: field rows from J0-2, v-rows and predictor rows from J0-1
  auto a = [&](int J) { return ta[(J - J0 + 2) * CW + c]; };
  auto vp = [&](int J) { return tvp[(J - J0 + 1) * CW + c]; };
  auto vm = [&](int J) { return tvm[(J - J0 + 1) * CW + c]; };
  auto aq = [&](int J) { return taq[(J - J0 + 1) * CW + c]; };
  auto ap = [&](int J) { return tap[(J - J0 + 1) * CW + c]; };
  // the field (rows outside -1..nj+1 are never read) and the velocities
  for (int r = r0; r < RA; r += RS) {
    const int J = J0 - 2 + r;
    ta[r * CW + c] = (J >= -1 && J <= nj + 1) ? T(A[ix2(d, J, I)]) : T(0.);
  }
  for (int r = r0; r < RV; r += RS) {
    const int J = J0 - 1 + r;
    if (J < 0 || J > nj + 1) continue;
    double v2;
    if (which == AV_HDRY) v2 = (J < 1 || J > nj) ? 0. : .5 * (d.V[ix3(d, K, J, I)] + d.V[ix3(d, K - 1, J, I)]);
    else v2 = d.V[ix3(d, K, J, I)];
    const double mi = d.minv_v[J];
    tvm[r * CW + c] = T(dmin(0., v2 * mi));
    tvp[r * CW + c] = T(dmax(0., v2 * mi));
  }
  __syncthreads();
  // smoothness terms and predictor on rows J0-1 .. J0+MER_TJ within 0..nj
  for (int r = r0; r < RP; r += RS) {
    const int J = J0 - 1 + r;
    if (J < 0 || J > nj) continue;
    T t;
    if (J == 0) t = fabs(-a(0) + a(1)) + ep;
    else if (J == nj) t = fabs(a(J - 1) - a(J)) + ep;
    else t = fabs(a(J - 1) - T(2.) * a(J) + a(J + 1)) + ep;
    taq[r * CW + c] = t * t;
    const T f0 = (J < 1) ? T(0.) : vp(J) * a(J - 1) + vm(J) * a(J);
    const T f1 = (J + 1 > nj) ? T(0.) : vp(J + 1) * a(J) + vm(J + 1) * a(J + 1);
    tap[r * CW + c] = a(J) + (f0 - f1) * T(d.mn[2 * J + 1]) * DT;
  }
  __syncthreads();
  // corrected flux on v-rows J0 .. J0+MER_TJ within 1..nj
  for (int r = r0; r <= MER_TJ; r += RS) {
    const int J = J0 + r;
    if (J < 1 || J > nj) continue;
    T VP = vp(J), VM = vm(J), APj = ap(J), APm = ap(J - 1), Am = a(J - 1), Aj = a(J);
    T fc = T(.5) * (VP * (APj + Am) + VM * (APm + Aj));
    T vhp = sqrt(VP * vp(J - 1)), vhm = -sqrt(VM * vm(J + 1));
    T mu = (VP - VM) * T(d.mn[2 * J]) * DT, al = (T(1.) + mu) / T(6.);
    T q0 = aq(J - 1), q1 = aq(J);
    T gp = q0 / (q0 + (Am - amin) * (Aj - amin));
    gp = gp * gp;
    T gm = q1 / (q1 + (Am - amin) * (Aj - amin));
    gm = gm * gm;
    T bp = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gp, bm = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gm;
    T bhp = T(1.) - gp, bhm = T(1.) - gm;
    T d1J = (APj - Am);
    T d1m = (J - 1 == 0) ? T(0.) : APm - a(J - 2);
    T d2m = APm - a(J);
    T d2J = (J == nj) ? T(0.) : APj - a(J + 1);
    tff[r * CW + c] = fc + -al * (VP * bp * d1J - vhp * bhp * d1m + VM * bm * d2m - vhm * bhm * d2J);
  }
  __syncthreads();
  // update on the tile's rows: the FP64 field plus the flux divergence
  const Plane<double> sA{d.sA + so + o};
  for (int r = r0; r < MER_TJ; r += RS) {
    const int J = J0 + r;
    if (J > nj) break;
    const T f0 = (J >= 1) ? tff[r * CW + c] : T(0.), f1 = (J + 1 <= nj) ? tff[(r + 1) * CW + c] : T(0.);
    sA[ix2(d, J, I)] = old_value(a(J), &A[ix2(d, J, I)]) + (double)((f0 - f1) * T(d.mn[2 * J + 1]) * DT);
  }
}

// --------------------------------------------------------------- zonal
// The zonal pass of row J by its ni/4 lanes, a lane holding the four points
// I = 1 + lane + q ni/4: a is the plane as the meridional pass left it (sA),
// y receives the row's result.  The row is rounded to the flux type, zonally
// filtered where it lies in the filter band, and staged in LDS with its pads
// beside the velocity u/n; first-guess flux, predictor and corrected flux
// follow on all lanes, periodic in I.  The filter runs here, on the row in registers, rather than
// in a launch of its own over a copy: the copy was a write and two reads of
// every field, and a wavefront without a row in the band skips the transform.
// Three row arrays: field, velocity (split by sign where it is used; the
// corrected flux overwrites it once every lane has read it) and predictor
// (before that, the filter's scratch); the first-guess flux is formed where
// the predictor needs it (twice per cell, by the same expression).
// the velocity on u-row J: U of the interface for unity and theta, the mean
// of the interfaces above and below for hdry (whose pads are the points they
// copy)
__device__ __forceinline__ double adv_u(const MemberDesc &d, bool layer, int K, int J, int I) {
  const Plane<const double> u{d.U + (size_t)K * d.N2};
  if (!layer) return u[ix2(d, J, I)];
  const Plane<const double> up{d.U + (size_t)(K - 1) * d.N2};
  const uint32_t i = ix2(d, J, I < 1 ? I + d.ni : (I > d.ni ? I - d.ni : I));
  return .5 * (u[i] + up[i]);
}
template <bool WIDE, class T>
__device__ __forceinline__ void hsu_zonal_row(const MemberDesc &d, const RowMap &m, bool layer, int K, int J, bool filt, T amin,
                                              const Plane<const double> &a, double (&y)[4], T *A) {
  const int ni = d.ni, W = ni + 2;
  const double ninv = d.ninv_h[J];
  T *UV = A + W, *AP = A + 2 * W, *FF = UV;
  const T mn = T(d.mn[2 * J + 1]), DT = T(d.dt);
  auto wr = [ni](int I) { return I < 1 ? I + ni : (I > ni ? I - ni : I); };
  T x[4];
#pragma unroll
  for (int q = 0; q < 4; q++) x[q] = T(a[ix2(d, J, 1 + m.lane + m.stride * q)]);
  // (the velocity and the FP64 row are read behind the transform, which
  // needs the registers they would hold)
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, x, AP, J, 0, filt, m.lane);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    A[I] = x[q];
    UV[I] = T(adv_u(d, layer, K, J, I) * ninv);
  }
  if (m.lane == 0) {
    A[ni + 1] = x[0];
    UV[ni + 1] = T(adv_u(d, layer, K, J, ni + 1) * ninv);
  }
  if (m.lane == m.stride - 1) {
    A[0] = x[3];
    UV[0] = T(adv_u(d, layer, K, J, 0) * ninv);
  }
  row_sync<WIDE>();
  // T(min(0, x)) = min(0, T(x)): rounding is monotone and keeps zero
  auto UP = [UV](int I) { return tmax(T(0.), UV[I]); };
  auto UM = [UV](int I) { return tmin(T(0.), UV[I]); };
  auto FP = [&](int c) { return UP(c) * A[c - 1] + UM(c) * A[c]; };
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = 1 + m.lane + m.stride * q;
    AP[c] = A[c] + (FP(c) - FP(wr(c + 1))) * mn * DT;
  }
  row_sync<WIDE>();
  // a lane's four corrected fluxes (c = 1 + lane + q*stride) in registers
  T ffr[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = 1 + m.lane + q * m.stride;
    const int cm = wr(c - 1);
    T UPc = UP(c), UMc = UM(c), APc = AP[c], APm = AP[cm], Am = A[c - 1], Ac = A[c];
    T fc = T(.5) * (UPc * (APc + Am) + UMc * (APm + Ac));
    T d1c = APc - Am, d2c = APc - A[c + 1];
    T d1m = APm - A[cm - 1], d2m = APm - A[cm + 1];
    T uhp = sqrt(UPc * UP(c - 1)), uhm = -sqrt(UMc * UM(c + 1));
    T mu = (UPc - UMc) * mn * DT, al = (T(1.) + mu) / T(6.);
    T t0 = fabs(A[cm - 1] - T(2.) * A[cm] + A[cm + 1]) + T(1.e-10), q0 = t0 * t0;
    T t1 = fabs(A[c - 1] - T(2.) * A[c] + A[c + 1]) + T(1.e-10), q1 = t1 * t1;
    T gp = q0 / (q0 + (Am - amin) * (Ac - amin));
    gp = gp * gp;
    T gm = q1 / (q1 + (Am - amin) * (Ac - amin));
    gm = gm * gm;
    T bp = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gp, bm = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * gm;
    T bhp = T(1.) - gp, bhm = T(1.) - gm;
    ffr[q] = fc + -al * (UPc * bp * d1c - uhp * bhp * d1m + UMc * bm * d2m - uhm * bhm * d2c);
    // one point at a time: interleaved, the four need 192 VGPRs
    __builtin_amdgcn_sched_barrier(0);
  }
  row_sync<WIDE>();
#pragma unroll
  for (int q = 0; q < 4; q++) FF[1 + m.lane + q * m.stride] = ffr[q];
  row_sync<WIDE>();
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + q * m.stride;
    y[q] = a[ix2(d, J, I)] + (double)((ffr[q] - FF[wr(I + 1)]) * mn * DT);
  }
}
// the Akima scheme's zonal pass of one row, in the same form
template <bool WIDE, class T>
__device__ __forceinline__ void ak_zonal_row(const MemberDesc &d, const RowMap &m, bool layer, int K, int J, bool filt,
                                             const Plane<const double> &a, double (&y)[4], T *A);

// Zonal pass of a row group (1024/ni rows of plane K per block).  layer: hdry,
// stored with the restore_mass that follows the advection.  Otherwise theta
// and, before it by the same lanes, unity, whose result corrects theta
// (theta - old (unity - 1), old the theta of before the advection, still where
// the column pass read it) and is written nowhere.  The two go through one copy of the code (a
// loop): written out twice the transform's operands are kept from one to the
// other and cost a wave of occupancy.
template <bool WIDE, class T, bool AKIMA>
__device__ __forceinline__ void adv_zonal_rows(const MemberDesc &d, bool layer, int hv, T *sh) {
  const RowMap m = row_map(d.ni);
  const int K = 1 + blockIdx.y, Jr = blockIdx.x * m.rpb + m.g, ni = d.ni;
  const bool live = Jr <= d.nj;
  const int J = live ? Jr : 0;
  T *A = sh + (size_t)m.g * 3 * (ni + 2);
  const bool filt = live && d.rflag_h[J] != 0;
  const size_t o = (size_t)K * d.N2;
  double y[4], cor[4];  // the field's row; unity's advected row less 1
#pragma unroll 1
  for (int which = layer ? AV_HDRY : AV_P3;; which = AV_THETA) {
    const Plane<const double> a{d.sA + (size_t)which * d.N3 + o};
    if constexpr (AKIMA) ak_zonal_row<WIDE, T>(d, m, layer, K, J, filt, a, y, A);
    else hsu_zonal_row<WIDE, T>(d, m, layer, K, J, filt, layer ? T(d.h_min[K]) : T(0.), a, y, A);
    if (which != AV_P3) break;
#pragma unroll
    for (int q = 0; q < 4; q++) cor[q] = y[q] - 1.;
    row_sync<WIDE>();
  }
  if (!live) return;
  const Plane<double> out{(layer ? d.HDRY : d.THETA) + o};
  const Plane<const double> old{adv_in(d, AV_THETA, hv) + o};
  const double hmin = d.h_min[K];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    double v = y[q];
    if (layer) v = dmax(hmin, v);
    else v -= old[ix2(d, J, I)] * cor[q];
    out[ix2(d, J, I)] = v;
    if (I == ni) out[ix2(d, J, 0)] = v;
    if (I == 1) out[ix2(d, J, ni + 1)] = v;
  }
}
// blockIdx.z = member for unity with theta, members + member for hdry
template <bool WIDE, class T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_hsu_zonal(const MemberDesc *D, int mb, int nm, int hv) {
  extern __shared__ double sh_raw[];
  const bool layer = (int)blockIdx.z >= nm;
  const MemberDesc &d = D[mb + (int)blockIdx.z - (layer ? nm : 0)];
  const int which = layer ? AV_HDRY : AV_THETA;
  if (d.adv_akima[which] || 1 + (int)blockIdx.y < adv_kfirst(d, which)) return;  // uniform per block
  adv_zonal_rows<WIDE, T, false>(d, layer, hv, reinterpret_cast<T *>(sh_raw));
}

// ------------------------------------------------------------- Akima
// akima_advection (src/shared/epic_flux.c:1502-1924), the monotonized
// fourth-order centred scheme, in the same three passes and tiles as the
// predictor-corrector above: the difference dA of neighbouring values, the
// harmonic-mean slope dela = 2 dA- dA+ / (dA- + dA+) where both have one
// sign (0 otherwise), and the flux: the velocity times the edge value
// .5 (a- + a+) - (dela+ - dela-) / 6, each by the reference's expression.
// A block whose field takes the other scheme returns at once (uniform per
// block).
// The reference also runs the column pass on the pad rows J = -1 and nj+1,
// where W3 is zero and the pass changes nothing.
template <class T>
__device__ __forceinline__ T ak_dela(T d0, T d1) {
  const T tmp = d0 * d1;
  return (tmp > T(0.)) ? T(2.) * tmp / (d0 + d1) : T(0.);
}

// column pass: columns J = 0..nj, I = 1..ni in LDS tiles; the stages
// (differences, slopes, fluxes, update) run on all lanes over (column,
// level) pairs, separated by barriers (no recurrence in K)
template <class T>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) k_ak_vert(const MemberDesc *D, int mb, int nm, int C, int hv) {
  ADV_MEMBER;
  if (!d.adv_akima[which]) return;  // uniform per block
  extern __shared__ double lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);
  const int c = threadIdx.x % C, kk = threadIdx.x / C, KS = blockDim.x / C;
  const int col = blockIdx.x * C + c;
  const bool live = col < (d.nj + 1) * d.ni;
  const int J = live ? col >> d.nlogn : 0, I = live ? 1 + (col & (d.ni - 1)) : 1;
  const int nk = d.nk, L = nk + 2;
  const int layer = (which == AV_HDRY);
  const int kf = (which == AV_THETA) ? d.ks - 1 : 1;
  const T DT = T(d.dt);
  const double *dsi = d.dsgth_inv;
  double *out = adv_out(d, which);
  // the flux reuses the difference column once the slopes are formed
  T *wa = lds + c * L, *wv = lds + (C + c) * L, *da = lds + (2 * C + c) * L, *dl = lds + (3 * C + c) * L, *ff = da;
  if (live)
    for (int K = kk; K <= nk + 1; K += KS) {
      double x = 0., w = 0.;
      if (layer) {
        if (K >= kf && K <= nk) x = adv_value(d, which, K, ix3(d, K, J, I), hv);
        if (K >= kf - 1 && K <= nk) w = d.W3[ix3(d, K, J, I)];
      } else {
        if (K >= kf - 1 && K <= nk) x = adv_value(d, which, K, ix3(d, K, J, I), hv);
        if (K >= kf && K <= nk) w = (K == 1 || K == nk) ? 0. : .5 * (d.W3[ix3(d, K, J, I)] + d.W3[ix3(d, K - 1, J, I)]);
      }
      wa[K] = T(x);
      wv[K] = T(w);
    }
  __syncthreads();
  // differences: in a layer, da[K] = a[K] - a[K+1] on kf..nk-1 (0 at kf-1
  // and nk); on interfaces, da[K] = a[K-1] - a[K] on kf..nk
  if (live)
    for (int K = kf - 1 + kk; K <= nk; K += KS) {
      if (layer) da[K] = (K == kf - 1 || K == nk) ? T(0.) : wa[K] - wa[K + 1];
      else if (K >= kf) da[K] = wa[K - 1] - wa[K];
    }
  __syncthreads();
  if (live)
    for (int K = kf - 1 + kk; K <= nk; K += KS) {
      if (layer) {
        if (K >= kf) dl[K] = ak_dela(da[K], da[K - 1]);
      } else {
        dl[K] = (K == kf - 1 || K == nk) ? T(0.) : ak_dela(da[K], da[K + 1]);
      }
    }
  __syncthreads();
  // fluxes (mass_flux_top and mass_flux_bot are zero)
  if (live)
    for (int K = kf - 1 + kk; K <= nk + 1; K += KS) {
      if (layer) {
        if (K <= nk)
          ff[K] = (K == kf - 1 || K == nk) ? T(0.) : wv[K] * (T(.5) * (wa[K] + wa[K + 1]) - (dl[K] - dl[K + 1]) / T(6.));
      } else if (K >= kf) {
        ff[K] = (K == nk + 1) ? T(0.) : wv[K] * (T(.5) * (wa[K - 1] + wa[K]) - (dl[K - 1] - dl[K]) / T(6.));
      }
    }
  __syncthreads();
  if (live)
    for (int K = max(kf, adv_kfirst(d, which)) + kk; K <= nk; K += KS) {
      const size_t q = ix3(d, K, J, I);
      const double x = col_value(wa[K], d, which, K, q, hv);
      if (layer) out[q] = x + (double)((ff[K] - ff[K - 1]) * T(dsi[2 * K]) * DT);
      else out[q] = x + (double)((ff[K + 1] - ff[K]) * T(dsi[2 * K + 1]) * DT);
    }
}

// meridional pass: a tile of TJ rows x CW columns of one plane, with the
// field on rows J0-2..J0+TJ+1, the slopes on J0-1..J0+TJ, the velocity and
// the fluxes on v-rows J0..J0+TJ; the update goes to sA, as the
// predictor-corrector's does
template <class T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_ak_mer(const MemberDesc *D, int mb, int nm, int CW, int MER_TJ) {
  ADV_MEMBER;
  const int K = 1 + blockIdx.y;
  if (!d.adv_akima[which] || K < adv_kfirst(d, which)) return;  // uniform per block
  extern __shared__ double sh_raw[];
  T *sh = reinterpret_cast<T *>(sh_raw);
  const int nj = d.nj, nchunk = d.ni / CW;
  const int tile = blockIdx.x / nchunk, chunk = blockIdx.x - tile * nchunk;
  const int J0 = tile * MER_TJ, c = threadIdx.x % CW, r0 = threadIdx.x / CW, RS = blockDim.x / CW;
  const int I = 1 + chunk * CW + c;
  const int RA = MER_TJ + 4, RV = MER_TJ + 1, RD = MER_TJ + 2;
  T *ta = sh, *tv = ta + RA * CW, *tdl = tv + RV * CW, *tff = tdl + RD * CW;
  const size_t o = (size_t)K * d.N2;
  const Plane<const double> A{adv_out(d, which) + o};
  const T DT = T(d.dt);
  auto a = [&](int J) { return ta[(J - J0 + 2) * CW + c]; };
  auto dl = [&](int J) { return tdl[(J - J0 + 1) * CW + c]; };
  for (int r = r0; r < RA; r += RS) {
    const int J = J0 - 2 + r;
    ta[r * CW + c] = (J >= -1 && J <= nj + 1) ? T(A[ix2(d, J, I)]) : T(0.);
  }
  for (int r = r0; r < RV; r += RS) {
    const int J = J0 + r;
    double v2 = 0.;
    if (J >= 1 && J <= nj)
      v2 = (which == AV_HDRY) ? .5 * (d.V[ix3(d, K, J, I)] + d.V[ix3(d, K - 1, J, I)]) : d.V[ix3(d, K, J, I)];
    tv[r * CW + c] = T(v2);
  }
  __syncthreads();
  // slopes on rows 0..nj (zero elsewhere; the differences are zero outside
  // the rows 1..nj)
  auto dA = [&](int J) { return (J >= 1 && J <= nj) ? a(J) - a(J - 1) : T(0.); };
  for (int r = r0; r < RD; r += RS) {
    const int J = J0 - 1 + r;
    tdl[r * CW + c] = (J >= 0 && J <= nj) ? ak_dela(dA(J), dA(J + 1)) : T(0.);
  }
  __syncthreads();
  for (int r = r0; r < RV; r += RS) {
    const int J = J0 + r;
    T f = T(0.);
    if (J >= 1 && J <= nj) {
      const double mi = d.minv_v[J];
      f = tv[r * CW + c] * (T(.5) * (a(J) + a(J - 1)) - (dl(J) - dl(J - 1)) / T(6.)) * T(mi);
    }
    tff[r * CW + c] = f;
  }
  __syncthreads();
  const Plane<double> sA{d.sA + so + o};
  for (int r = r0; r < MER_TJ; r += RS) {
    const int J = J0 + r;
    if (J > nj) break;
    sA[ix2(d, J, I)] =
        old_value(a(J), &A[ix2(d, J, I)]) + (double)((tff[r * CW + c] - tff[(r + 1) * CW + c]) * T(d.mn[2 * J + 1]) * DT);
  }
}

// zonal pass of one row: the filtered row with its pads in LDS; slopes,
// fluxes and the update on all lanes of the row, periodic in I
template <bool WIDE, class T>
__device__ __forceinline__ void ak_zonal_row(const MemberDesc &d, const RowMap &m, bool layer, int K, int J, bool filt,
                                             const Plane<const double> &a, double (&y)[4], T *A) {
  const int ni = d.ni, W = ni + 2;
  T *DL = A + W, *FF = A + 2 * W;
  const T mn = T(d.mn[2 * J + 1]), DT = T(d.dt);
  const double ninv = d.ninv_h[J];
  auto wr = [ni](int I) { return I < 1 ? I + ni : (I > ni ? I - ni : I); };
  T x[4];
#pragma unroll
  for (int q = 0; q < 4; q++) x[q] = T(a[ix2(d, J, 1 + m.lane + m.stride * q)]);
  if (filter_any<WIDE>(filt)) filter_row_regs<WIDE>(d, x, FF, J, 0, filt, m.lane);
#pragma unroll
  for (int q = 0; q < 4; q++) A[1 + m.lane + m.stride * q] = x[q];
  if (m.lane == 0) A[ni + 1] = x[0];
  if (m.lane == m.stride - 1) A[0] = x[3];
  row_sync<WIDE>();
  // differences A(I) - A(I-1) on I = 1..ni, the pad of I = ni+1 that of I = 1
  auto dA = [&](int I) { return A[I] - A[I - 1]; };
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    DL[I] = ak_dela(dA(I), dA(wr(I + 1)));
  }
  row_sync<WIDE>();
  T f[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    f[q] = T(adv_u(d, layer, K, J, I)) * (T(.5) * (A[I] + A[I - 1]) - (DL[I] - DL[wr(I - 1)]) / T(6.)) * T(ninv);
    FF[I] = f[q];
  }
  row_sync<WIDE>();
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int I = 1 + m.lane + m.stride * q;
    y[q] = a[ix2(d, J, I)] + (double)((f[q] - FF[wr(I + 1)]) * mn * DT);
  }
}
template <bool WIDE, class T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_ak_zonal(const MemberDesc *D, int mb, int nm, int hv) {
  extern __shared__ double sh_raw[];
  const bool layer = (int)blockIdx.z >= nm;
  const MemberDesc &d = D[mb + (int)blockIdx.z - (layer ? nm : 0)];
  const int which = layer ? AV_HDRY : AV_THETA;
  if (!d.adv_akima[which] || 1 + (int)blockIdx.y < adv_kfirst(d, which)) return;  // uniform per block
  adv_zonal_rows<WIDE, T, true>(d, layer, hv, reinterpret_cast<T *>(sh_raw));
}

// restore_mass, one advection pass over all three fields of every member,
// restore_mass (src/shared/epic_timestep.c, src/shared/epic_flux.c); the mixed
// mode forms the fluxes in FP32.  Each scheme's launches run where some field
// of the bucket takes it.  set_p2etc(DONT_UPDATE_THETA) follows, with
// store_pgrad_vars.
template <class T>
static void advection_t(hipStream_t s, const Bucket &b) {
  const int hv = hv_fused(b) ? 1 : 0;
  const int ncol = (b.nj + 1) * b.ni, nz = ADV_FIELDS * b.nm;
  // columns per block: as many as keep the four LDS columns within 40 KB
  int C = 64;
  while (C > 16 && (size_t)4 * C * (b.nk + 2) * sizeof(double) > 40 * 1024) C /= 2;
  const int v = b.knob[KN_COLS_HSUV];
  if (v) C = knob_cols(v);
  const bool hsu = b.adv_schemes & 1, akima = b.adv_schemes & 2;
  const dim3 gv((ncol + C - 1) / C, 1, nz);
  if (hsu)
    LAUNCH(k_hsu_vert<T>, gv, dim3(knob_threads(v, b.nk + 2)), sizeof(T) * 4 * C * (b.nk + 2), s, b.D, b.mb, b.nm, C, hv);
  if (akima) LAUNCH(k_ak_vert<T>, gv, dim3(knob_threads(v, b.nk + 2)), sizeof(T) * 4 * C * (b.nk + 2), s, b.D, b.mb, b.nm, C, hv);
  const int TJ = b.knob[KN_ROWS_MER] ? b.knob[KN_ROWS_MER] : 4;
  const int CW = b.ni < 64 ? b.ni : 64, tiles = (b.nj + 1 + TJ - 1) / TJ;
  const dim3 gm(tiles * (b.ni / CW), b.nk, nz);
  if (hsu)
    LAUNCH(k_hsu_mer<T>, gm, dim3(256), sizeof(T) * CW * ((TJ + 4) + 2 * (TJ + 3) + 2 * (TJ + 2) + (TJ + 1)), s, b.D,
           b.mb, b.nm, CW, TJ);
  if (akima)
    LAUNCH(k_ak_mer<T>, gm, dim3(256), sizeof(T) * CW * ((TJ + 4) + 2 * (TJ + 1) + (TJ + 2)), s, b.D, b.mb, b.nm, CW,
           TJ);
  const int rpb = rows_per_block(b.ni);
  const dim3 gz((b.nj + 1 + rpb - 1) / rpb, b.nk, 2 * b.nm);
  if (hsu) ROWS_LAUNCH(b, "k_hsu_zonal<T>", (k_hsu_zonal<true, T>), (k_hsu_zonal<false, T>), gz, dim3(256), sizeof(T) * rpb * 3 * (b.ni + 2), s, b.D, b.mb, b.nm, hv);
  if (akima) ROWS_LAUNCH(b, "k_ak_zonal<T>", (k_ak_zonal<true, T>), (k_ak_zonal<false, T>), gz, dim3(256), sizeof(T) * rpb * 3 * (b.ni + 2), s, b.D, b.mb, b.nm, hv);
}
void L_advection(hipStream_t s, const Bucket &b) {
  if (b.mixed) advection_t<float>(s, b);
  else advection_t<double>(s, b);
}

}  // namespace epic
