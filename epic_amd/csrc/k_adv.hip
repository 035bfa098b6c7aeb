// k_adv.hip -- flux-form predictor-corrector advection of Hsu & Arakawa as
// modified by Konor & Arakawa (hsu_advection, src/shared/epic_flux.c:652-1488),
// the monotonized fourth-order centred scheme offered beside it (Akima,
// akima_advection, src/shared/epic_flux.c:1502-1924), and their driver
// (advection, src/shared/epic_flux.c:346-637).
//
// Directions are split as in the reference: vertical column pass, then a
// meridional pass on every level, then a zonal pass on a zonally filtered
// copy.  The column and meridional passes hold a few cells of a line with
// their reach in a lane's registers (Akima's: LDS tiles), the zonal pass works
// on LDS rows; every intermediate value is formed by the same expression as
// in the reference, so nothing changes but where it is computed.
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
// preceding unity call.  w_a is unity before its advection, 1 everywhere; wm
// meets the predicted change behind that face, which is 0 there.
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

// The advection passes are templated on the arithmetic type T of the fluxes:
// double reproduces the reference operation for operation; float is the
// mixed mode's (the fields stay FP64: each update adds the FP32 flux
// divergence to the FP64 value).

// x / 6, correctly rounded, for finite x of ordinary size: the product with
// the rounded reciprocal is within an ulp, and one fused correction of its
// exact remainder rounds it right (Markstein, IBM J. Res. Dev. 34, 1990)
__device__ __forceinline__ double div6(double x) {
  const double q = x * (1. / 6.);
  return fma(fma(-6., q, x), 1. / 6., q);
}
__device__ __forceinline__ float div6(float x) {
  const float q = x * (1.f / 6.f);
  return fmaf(fmaf(-6.f, q, x), 1.f / 6.f, q);
}

// The corrected flux through the face between cells m and j; v > 0 carries m
// into j.  The reference forms it from v split by sign, as the sum of a
// positive and a negative part of which one is zero; here the part that is
// not is formed alone, with the donor's (D) and the receiver's (R) values
// picked by v's sign: the same operations in the same order, half the
// divisions and square roots.  (Only a zero's sign, and how many cells a NaN
// spreads in one pass, can differ.)  dh: the predicted change from the cell
// behind the donor to the donor; nb: the velocity of the face behind it; qD:
// its smoothness term; prod: (a_D - min)(a_R - min); c: the metric factor of
// the Courant number.
template <class T>
__device__ __forceinline__ T hsu_flux(T v, T aD, T pR, T dh, T qD, T nb, T prod, T c, T DT) {
  const T fc = T(.5) * (v * (pR + aD));
  const T x = v * nb;
  const T vh = copysign(sqrt(x < T(0.) ? T(0.) : x), v);
  const T al = div6(T(1.) + fabs(v) * c * DT);
  T g = qD / (qD + prod);
  g = g * g;
  const T b = T(1.) + (T(1.) / (T(2.) * al) - T(1.)) * g;
  return fc + -al * (v * b * (pR - aD) - vh * (T(1.) - g) * dh);
}

// The FP64 value a pass updates: the staged copy itself when the pass
// computes in FP64 (the same bits), else a re-read of the FP64 field
__device__ __forceinline__ double old_value(double staged, const double *) { return staged; }
__device__ __forceinline__ double old_value(float, const double *p) { return *p; }
__device__ __forceinline__ double col_value(double staged, const MemberDesc &, int, int, size_t, int) { return staged; }
__device__ __forceinline__ double col_value(float, const MemberDesc &d, int which, int K, size_t q, int hv) {
  return adv_value(d, which, K, q, hv);
}

// ------------------------------------------------------------ vertical
// A lane takes one column (J = 0..nj, I = 1..ni) and KC of its levels in
// registers, with the two levels above and below them that the K-stencils
// (first-guess flux, predictor, centred flux, limiter correction, update)
// reach: cells K0-2..K0+KC+1 and the velocities of the faces K0-2..K0+KC,
// face k lying between cells k and k+1 (for unity and theta, whose cells are
// the interfaces, the mean of W3 above and below).  Every load is issued
// before the first flux; nothing passes through LDS and the level's metric
// terms are scalar.  Cells and faces outside the column are formed from
// whatever the clamped loads gave and replaced.
// (As stages over an LDS column tile with barriers between, the addresses
// and waits were most of it: 1730 us against 681 at 1024x512x64, 23.2 against
// 14.7 at 256x128x20, both FP64.)
// LAYER: hdry.  EDGE: the reach K0-2..K0+KC+1 touches the top or the bottom
// (interior chunks carry none of the tests).
template <class T, int KC, bool LAYER, bool EDGE>
__device__ __forceinline__ void hsu_vert_cells(const MemberDesc &d, int which, int hv, int K0, int kf, int kout, uint32_t i) {
  const int nk = d.nk;
  const T ep = T(1.e-10), DT = T(d.dt);
  const double *dsi = d.dsgth_inv + (LAYER ? 0 : 1);  // [2k]: of cell k; [2k+1]: of face k
  const double *in = adv_in(d, which, hv);
  auto lev = [&](int k, int k0) { return EDGE ? min(max(k, k0), nk) : k; };
  double f[KC + 4], w[KC + 4];  // the field on cells K0-2 .., W3
#pragma unroll
  for (int r = 0; r < KC + 4; r++) f[r] = 1.;  // unity
  if (LAYER || which == AV_THETA) {
#pragma unroll
    for (int r = 0; r < KC + 4; r++) {
      const int k = lev(K0 - 2 + r, LAYER ? 1 : kf - 1);
      // theta above its first advected level is the field's own
      const double *x = (EDGE && !LAYER && k < d.ks - 1) ? d.THETA : in;
      f[r] = Plane<const double>{x + (size_t)k * d.N2}[i];
    }
  }
#pragma unroll
  for (int r = 0; r < KC + (LAYER ? 3 : 4); r++) w[r] = Plane<const double>{d.W3 + (size_t)lev(K0 - 2 + r, 0) * d.N2}[i];
  if (LAYER) {
#pragma unroll
    for (int r = 0; r < KC + 4; r++) f[r] = dmax(d.h_min[lev(K0 - 2 + r, 1)], f[r]);
  } else if (EDGE && which == AV_THETA) {  // the reference's static work column holds unity there
#pragma unroll
    for (int r = 0; r < KC + 4; r++)
      if (K0 - 2 + r < kf - 1) f[r] = 1.;
  }
  __builtin_amdgcn_sched_barrier(0);  // every load before the first flux
  // from here on one face after another, each with the cell it enters
  T a[KC + 4], v[KC + 3], g0[KC + 3], p[KC + 2], q[KC + 2], F[KC + 1];
#pragma unroll
  for (int r = 0; r < KC + 4; r++) a[r] = T(f[r]);
  // the velocity of face k = K0-2+r and its first-guess flux (none through the
  // bottom, nor through a layer's top)
  auto guess = [&](int r) {
    const int k = K0 - 2 + r;
    v[r] = T(LAYER ? w[r] : .5 * (w[r + 1] + w[r]));
    if (EDGE && !LAYER && (k < max(kf - 1, 1) || k >= nk - 1)) v[r] = T(0.);
    g0[r] = v[r] * (v[r] > T(0.) ? a[r + 1] : a[r]);
    if (EDGE && (k >= nk || (LAYER && k <= 0))) g0[r] = T(0.);
  };
  // predictor and smoothness term of cell k = K0-1+r
  auto cell = [&](int r) {
    const int k = K0 - 1 + r;
    p[r] = a[r + 1] + (g0[r + 1] - g0[r]) * T(dsi[2 * lev(k, 0)]) * DT;
    if (EDGE && !LAYER && k == kf - 1) p[r] = a[r + 1];
    T t = a[r + 2] - T(2.) * a[r + 1] + a[r];
    if (EDGE && k == (LAYER ? 1 : 0)) t = a[r + 2] - a[r + 1];
    else if (EDGE && k == nk) t = -a[r + 1] + a[r];
    t = fabs(t) + ep;
    q[r] = t * t;
  };
  double *out = adv_out(d, which);
  guess(0);
  guess(1);
  cell(0);
#pragma unroll
  for (int r = 0; r < KC + 1; r++) {
    // corrected flux through face k: cell j = k above, m = k+1 below
    const int k = K0 - 1 + r, kk = EDGE ? min(k, nk - 1) : k;
    guess(r + 2);
    cell(r + 1);
    const bool up = v[r + 1] > T(0.);
    const T aj = a[r + 1], am = a[r + 2];
    const T prod = LAYER ? (am - T(d.h_min[kk + 1])) * (aj - T(d.h_min[EDGE ? max(kk, 1) : kk])) : am * aj;
    // the predicted change behind the donor; none at the column's ends
    T dm = p[r + 1] - a[r + 3], dj = p[r] - a[r];
    if (EDGE && k + 1 == nk) dm = T(0.);
    if (EDGE && k == (LAYER ? 1 : kf - 1)) dj = T(0.);
    F[r] = hsu_flux<T>(v[r + 1], up ? am : aj, up ? p[r] : p[r + 1], up ? dm : dj, up ? q[r + 1] : q[r],
                       up ? v[r + 2] : v[r], prod, T(dsi[2 * kk + 1]), DT);
    if (EDGE && (k >= nk || (LAYER && k <= 0))) F[r] = T(0.);
    if (r > 0 && !(EDGE && (k < kout || k > nk)))
      Plane<double>{out + (size_t)k * d.N2}[i] = f[r + 1] + (double)((F[r] - F[r - 1]) * T(dsi[2 * k]) * DT);
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <class T, int KC>
__global__ void __launch_bounds__(256) k_hsu_vert(const MemberDesc *D, int mb, int nm, int hv) {
  ADV_MEMBER;
  const int nk = d.nk, K0 = 1 + (int)blockIdx.y * KC;
  const bool layer = (which == AV_HDRY);
  const int kf = (which == AV_THETA) ? d.ks - 1 : 1;
  // unity's levels above k_sigma-1 serve their neighbours only
  const int kout = layer ? 1 : max(kf, d.ks - 1);
  if (d.adv_akima[which] || K0 + KC <= kout) return;  // uniform per block
  const int col = blockIdx.x * TPB + threadIdx.x;
  if (col >= (d.nj + 1) * d.ni) return;
  const uint32_t i = ix2(d, col >> d.nlogn, 1 + (col & (d.ni - 1)));
  const bool edge = K0 - 2 < max(kout, 2) || K0 + KC + 1 >= nk;  // uniform per block
  if (layer) {
    if (edge) hsu_vert_cells<T, KC, true, true>(d, which, hv, K0, kf, kout, i);
    else hsu_vert_cells<T, KC, true, false>(d, which, hv, K0, kf, kout, i);
  } else {
    if (edge) hsu_vert_cells<T, KC, false, true>(d, which, hv, K0, kf, kout, i);
    else hsu_vert_cells<T, KC, false, false>(d, which, hv, K0, kf, kout, i);
  }
}

// ---------------------------------------------------------- meridional
// A lane takes one longitude of a plane and TJ rows in registers, with the
// rows around them as the column pass does: the field on rows J0-2..J0+TJ+1,
// the velocity v/m on v-rows J0-1..J0+TJ+1 (v-row J lies between rows J-1 and
// J), predictor and smoothness terms on rows J0-1..J0+TJ and the corrected
// flux on v-rows J0..J0+TJ; the halo rows are formed again by the
// neighbouring lane (the same values).  SROW: a wavefront lies in one row
// tile, whose metric terms are scalar.  The update goes to sA.
// (From an LDS tile of 64 columns: 1700 us against 680 at 1024x512x64, 26.6
// against 14.6 at 256x128x20, both FP64; 423 vector instructions a cell.)
// EDGE: the reach touches a pole (the tiles between carry none of the tests).
template <class T, int TJ, bool EDGE>
__device__ __forceinline__ void hsu_mer_cells(const MemberDesc &d, int which, int K, int J0, int I) {
  const int nj = d.nj;
  const bool layer = (which == AV_HDRY);
  const size_t o = (size_t)K * d.N2;
  const Plane<const double> A{adv_out(d, which) + o}, V{d.V + o}, VU{d.V + o - d.N2};
  const T amin = layer ? T(d.h_min[K]) : T(0.), DT = T(d.dt), ep = T(1.e-10);
  auto row = [&](int J, int lo, int hi) { return EDGE ? min(max(J, lo), hi) : J; };
  double f[TJ + 4], v64[TJ + 3];
#pragma unroll
  for (int r = 0; r < TJ + 4; r++) f[r] = A[ix2(d, row(J0 - 2 + r, -1, nj + 1), I)];
#pragma unroll
  for (int r = 0; r < TJ + 3; r++) v64[r] = V[ix2(d, row(J0 - 1 + r, 0, nj + 1), I)];
  if (layer) {
#pragma unroll
    for (int r = 0; r < TJ + 3; r++) {
      const int J = J0 - 1 + r;
      v64[r] = .5 * (v64[r] + VU[ix2(d, row(J, 0, nj + 1), I)]);
      if (EDGE && (J < 1 || J > nj)) v64[r] = 0.;
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load before the first flux
  T a[TJ + 4], v[TJ + 3], g0[TJ + 3], p[TJ + 2], q[TJ + 2], F[TJ + 1];
#pragma unroll
  for (int r = 0; r < TJ + 4; r++) a[r] = T(f[r]);
  auto guess = [&](int r) {
    const int J = J0 - 1 + r;
    v[r] = T(v64[r] * d.minv_v[row(J, 0, nj + 1)]);
    g0[r] = v[r] * (v[r] > T(0.) ? a[r] : a[r + 1]);
    if (EDGE && (J < 1 || J > nj)) g0[r] = T(0.);
  };
  auto cell = [&](int r) {
    const int J = J0 - 1 + r;
    p[r] = a[r + 1] + (g0[r] - g0[r + 1]) * T(d.mn[2 * row(J, 0, nj) + 1]) * DT;
    T t = a[r] - T(2.) * a[r + 1] + a[r + 2];
    if (EDGE && J == 0) t = -a[r + 1] + a[r + 2];
    else if (EDGE && J == nj) t = a[r] - a[r + 1];
    t = fabs(t) + ep;
    q[r] = t * t;
  };
  const Plane<double> sA{d.sA + (size_t)which * d.N3 + o};
  guess(0);
  guess(1);
  cell(0);
#pragma unroll
  for (int r = 0; r < TJ + 1; r++) {
    const int J = J0 + r;
    guess(r + 2);
    cell(r + 1);
    const bool up = v[r + 1] > T(0.);
    const T am = a[r + 1], aj = a[r + 2];
    // the predicted change behind the donor; none at the poles
    T dm = p[r] - a[r], dj = p[r + 1] - a[r + 3];
    if (EDGE && J == 1) dm = T(0.);
    if (EDGE && J == nj) dj = T(0.);
    F[r] = hsu_flux<T>(v[r + 1], up ? am : aj, up ? p[r + 1] : p[r], up ? dm : dj, up ? q[r] : q[r + 1],
                       up ? v[r] : v[r + 2], (am - amin) * (aj - amin), T(d.mn[2 * row(J, 0, nj)]), DT);
    if (EDGE && (J < 1 || J > nj)) F[r] = T(0.);
    if (r > 0 && !(EDGE && J - 1 > nj))
      sA[ix2(d, J - 1, I)] = f[r + 1] + (double)((F[r - 1] - F[r]) * T(d.mn[2 * J - 1]) * DT);
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <class T, int TJ, bool SROW>
__global__ void __launch_bounds__(256) k_hsu_mer(const MemberDesc *D, int mb, int nm) {
  const int which = (int)blockIdx.z / nm;
  const MemberDesc &d = D[mb + (int)blockIdx.z - which * nm];
  const int K = 1 + blockIdx.y;
  if (d.adv_akima[which] || K < adv_kfirst(d, which)) return;  // uniform per block
  const int t0 = blockIdx.x * TPB + threadIdx.x, tile = t0 >> d.nlogn;
  const int J0 = TJ * (SROW ? __builtin_amdgcn_readfirstlane(tile) : tile), I = 1 + (t0 & (d.ni - 1));
  if (J0 > d.nj) return;
  if (SROW && J0 >= 2 && J0 + TJ < d.nj) hsu_mer_cells<T, TJ, false>(d, which, K, J0, I);
  else hsu_mer_cells<T, TJ, true>(d, which, K, J0, I);
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
// Three row arrays: field, velocity (the
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
  auto FP = [&](int c) { return UV[c] * (UV[c] > T(0.) ? A[c - 1] : A[c]); };
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = 1 + m.lane + m.stride * q;
    AP[c] = A[c] + (FP(c) - FP(wr(c + 1))) * mn * DT;
  }
  row_sync<WIDE>();
  // a lane's four corrected fluxes (c = 1 + lane + q*stride) in registers:
  // the face between cells cm = c-1 and c
  T ffr[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = 1 + m.lane + q * m.stride, cm = wr(c - 1);
    const T u = UV[c];
    const bool up = u > T(0.);
    const int e = up ? cm : c;  // the donor
    const T aD = A[e], aR = A[up ? c : cm], aW = A[e - 1], aE = A[e + 1];
    const T t = fabs(aW - T(2.) * aD + aE) + T(1.e-10);
    ffr[q] = hsu_flux<T>(u, aD, AP[up ? c : cm], AP[e] - (up ? aW : aE), t * t, UV[up ? c - 1 : c + 1],
                         (aD - amin) * (aR - amin), mn, DT);
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
template <class T, int KC>
static void hsu_vert(hipStream_t s, const Bucket &b, int hv) {
  LAUNCH_AS("k_hsu_vert<T>", (k_hsu_vert<T, KC>), dim3(((b.nj + 1) * b.ni + TPB - 1) / TPB, (b.nk + KC - 1) / KC, ADV_FIELDS * b.nm),
            dim3(TPB), 0, s, b.D, b.mb, b.nm, hv);
}
template <class T, int TJ>
static void hsu_mer(hipStream_t s, const Bucket &b) {
  const int tiles = (b.nj + TJ) / TJ;
  const dim3 g((tiles * b.ni + TPB - 1) / TPB, b.nk, ADV_FIELDS * b.nm);
  if (b.ni >= 64) LAUNCH_AS("k_hsu_mer<T>", (k_hsu_mer<T, TJ, true>), g, dim3(TPB), 0, s, b.D, b.mb, b.nm);
  else LAUNCH_AS("k_hsu_mer<T>", (k_hsu_mer<T, TJ, false>), g, dim3(TPB), 0, s, b.D, b.mb, b.nm);
}
template <class T>
static void advection_t(hipStream_t s, const Bucket &b) {
  const int hv = hv_fused(b) ? 1 : 0;
  const int ncol = (b.nj + 1) * b.ni, nz = ADV_FIELDS * b.nm;
  // columns per block: as many as keep the four LDS columns within 40 KB
  int C = 64;
  while (C > 16 && ak_col_lds(b, C) > 40 * 1024) C /= 2;
  const int v = b.knob[KN_COLS_HSUV];
  if (v) C = knob_cols(v);
  const bool hsu = b.adv_schemes & 1, akima = b.adv_schemes & 2;
  const dim3 gv((ncol + C - 1) / C, 1, nz);
  // More cells per lane form fewer halo cells again and leave fewer lanes: 8
  // of each from 2^22 points up (16.51 against 16.66 ms a step with 4 at
  // 1024x512x64, no difference at 2^22), 4 below (473 against 476 us with 8 at
  // 256x128x20, 156 against 159 us at 32x19x7)
  const bool big = (size_t)b.ni * (b.nj + 1) * b.nk * b.nm >= ((size_t)1 << 22);
  if (hsu) {
    if (big) hsu_vert<T, 8>(s, b, hv);
    else hsu_vert<T, 4>(s, b, hv);
  }
  if (akima) LAUNCH(k_ak_vert<T>, gv, dim3(knob_threads(v, b.nk + 2)), sizeof(T) * 4 * C * (b.nk + 2), s, b.D, b.mb, b.nm, C, hv);
  const int kn = b.knob[KN_ROWS_MER], TJ = kn ? kn : 4, TJH = kn ? kn : big ? 8 : 4;
  const int CW = b.ni < 64 ? b.ni : 64, tiles = (b.nj + 1 + TJ - 1) / TJ;
  const dim3 gm(tiles * (b.ni / CW), b.nk, nz);
  if (hsu) {
    if (TJH == 2) hsu_mer<T, 2>(s, b);
    else if (TJH == 4) hsu_mer<T, 4>(s, b);
    else hsu_mer<T, 8>(s, b);
  }
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
