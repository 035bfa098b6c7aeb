// filter_row.h -- the polar-filter transform shared by the kernels that
// filter rows: the NR real FFT of src/shared/epic_funcs_util.c:4023-4135
// (four1 stages and the realft split step, with the twiddles of the
// reference's recurrences tabulated on the host; the stage-s twiddle m is
// complex entry 2^s - 1 + m), one butterfly per lane,
// and filter_row_regs(), which filters one latitude row held by its lanes
// inside a consumer kernel (src/shared/epic_adjust.c:102-242, TWODIM).
#pragma once
#include "dev_common.h"

namespace epic {

__device__ __forceinline__ int brev(int k, int bits) { return bits ? (int)(__brev((unsigned)k) >> (32 - bits)) : 0; }

// Barrier between the transform stages of one row.  A row's ni/4 lanes lie
// in one wavefront when ni <= 256, and rows never exchange data, so a
// wavefront-level barrier suffices there; larger rows (WIDE, ni > 256) span
// waves.  WIDE is a template argument of every row kernel: tested at each
// barrier, it had the compiler duplicate the code behind it (the zonal
// advection pass took 134 VGPRs instead of 78).
template <bool WIDE>
__device__ __forceinline__ void row_sync() {
  if constexpr (WIDE) __syncthreads();
  else wave_sync();
}

// one radix-2 butterfly of the reference's four1 on (xr, xi) and (yr, yi)
// with twiddle (wr, wi), in its operation order
template <class T>
__device__ __forceinline__ void bfly(T &xr, T &xi, T &yr, T &yi, T wr, T wi) {
  const T tr = wr * yr - wi * yi;
  const T ti = wr * yi + wi * yr;
  yr = xr - tr;
  yi = xi - ti;
  xr += tr;
  xi += ti;
}

// twiddle tables and field views of a storage type
template <class T> __device__ __forceinline__ const T *tw_fwd(const MemberDesc &d);
template <class T> __device__ __forceinline__ const T *tw_inv(const MemberDesc &d);
template <class T> __device__ __forceinline__ const T *tr_fwd(const MemberDesc &d);
template <class T> __device__ __forceinline__ const T *tr_inv(const MemberDesc &d);
template <> __device__ __forceinline__ const double *tw_fwd<double>(const MemberDesc &d) { return d.tw_f; }
template <> __device__ __forceinline__ const double *tw_inv<double>(const MemberDesc &d) { return d.tw_i; }
template <> __device__ __forceinline__ const double *tr_fwd<double>(const MemberDesc &d) { return d.tr_f; }
template <> __device__ __forceinline__ const double *tr_inv<double>(const MemberDesc &d) { return d.tr_i; }
template <> __device__ __forceinline__ const float *tw_fwd<float>(const MemberDesc &d) { return d.tw_f32; }
template <> __device__ __forceinline__ const float *tw_inv<float>(const MemberDesc &d) { return d.tw_i32; }
template <> __device__ __forceinline__ const float *tr_fwd<float>(const MemberDesc &d) { return d.tr_f32; }
template <> __device__ __forceinline__ const float *tr_inv<float>(const MemberDesc &d) { return d.tr_i32; }

// Where complex element p of a row lies in the transform's scratch: the low
// four bits of its place mixed with the next four.  In natural order the
// bit-reversed stores of 64 lanes fall 16 elements (256 bytes, all 64 banks)
// apart at ni = 1024 and the points of the first stage pairs 4 or 16: waiting
// for the same banks was over a third of the row kernels' time.  A permutation
// of each 16 elements, linear over exclusive or: swz(p ^ q) = swz(p) ^ swz(q).
// FP64 steps before and after: 256x128x20 429 and 413 us, 23 members of
// 128x51x13 945 and 920, 1024x512x64 14.39 and 14.26 ms; k_hv4, 1024x512x64:
// 853 and 750 us.
__device__ __forceinline__ int swz(int p) { return p ^ ((p >> 4) & 15); }
// the same for value e of the row (element e/2, real or imaginary)
__device__ __forceinline__ int swz_val(int e) { return 2 * swz(e >> 1) + (e & 1); }

// unit `lane` (of n/8) of the stages s and s+1, h = 2^s, on a row in LDS, its elements
// at swz: the
// four points p, p+h, p+2h, p+3h go through stage s as (p, p+h) and
// (p+2h, p+3h) and through stage s+1 as (p, p+2h) and (p+h, p+3h), in
// registers
template <class T>
__device__ __forceinline__ void four1_pair(T *buf, int s, int lane, const T *tw) {
  const int half = 1 << s, mm = lane & (half - 1), g = lane >> s;
  // (mm + 4 half g has zeros where half and 2 half have their bit)
  const int i0 = 2 * swz(mm + g * 4 * half), i1 = i0 ^ (2 * swz(half)), i2 = i0 ^ (2 * swz(2 * half)),
            i3 = i0 ^ (2 * swz(3 * half));
  T x0r = buf[i0], x0i = buf[i0 + 1], x1r = buf[i1], x1i = buf[i1 + 1];
  T x2r = buf[i2], x2i = buf[i2 + 1], x3r = buf[i3], x3i = buf[i3 + 1];
  const int ka = half - 1 + mm, kb = 2 * half - 1 + mm;
  const T ar = tw[2 * ka], ai = tw[2 * ka + 1];
  const T br = tw[2 * kb], bi = tw[2 * kb + 1], cr = tw[2 * (kb + half)], ci = tw[2 * (kb + half) + 1];
  bfly(x0r, x0i, x1r, x1i, ar, ai);
  bfly(x2r, x2i, x3r, x3i, ar, ai);
  bfly(x0r, x0i, x2r, x2i, br, bi);
  bfly(x1r, x1i, x3r, x3i, cr, ci);
  buf[i0] = x0r;
  buf[i0 + 1] = x0i;
  buf[i1] = x1r;
  buf[i1 + 1] = x1i;
  buf[i2] = x2r;
  buf[i2 + 1] = x2i;
  buf[i3] = x3r;
  buf[i3 + 1] = x3i;
}
// unit `lane` (of n/4) of one stage s: the odd last one
template <class T>
__device__ __forceinline__ void four1_last(T *buf, int s, int lane, const T *tw) {
  const int half = 1 << s, g = lane >> s, mm = lane & (half - 1), k = half - 1 + mm;
  const int i0 = 2 * swz(mm + g * 2 * half), j0 = i0 ^ (2 * swz(half));
  T xr = buf[i0], xi = buf[i0 + 1], yr = buf[j0], yi = buf[j0 + 1];
  bfly(xr, xi, yr, yi, tw[2 * k], tw[2 * k + 1]);
  buf[i0] = xr;
  buf[i0 + 1] = xi;
  buf[j0] = yr;
  buf[j0 + 1] = yi;
}

// complex radix-2 stages on buf[0..n) (n doubles = n/2 complex, at swz), in the
// reference's stage order.  Stages go two at a time: a lane loads the four
// points p, p+h, p+2h, p+3h (h = 2^s) into registers, applies stage s to
// (p, p+h) and (p+2h, p+3h) and stage s+1 to (p, p+2h) and (p+h, p+3h), and
// stores them: every point sees the same butterflies in the same order as
// with one stage per pass, with half the LDS round trips and barriers.  n/8
// lanes take part in a pair of stages; an odd last stage runs one butterfly
// per lane on n/4 lanes.
template <bool WIDE, class T>
__device__ __forceinline__ void four1_stages(T *buf, int n, int lane, const T *tw, bool active) {
  int S = 0;
  while ((2 << S) < n) S++;  // stages s with 2 << s < n
  int s = 0;
  for (; s + 1 < S; s += 2) {
    if (active && lane < (n >> 3)) four1_pair(buf, s, lane, tw);
    row_sync<WIDE>();
  }
  if (s < S) {
    if (active) four1_last(buf, s, lane, tw);
    row_sync<WIDE>();
  }
}

// One lane's four values between the forward and the inverse transform: the
// split step of the forward real transform, the filter's gains and the split
// step of the inverse.  Unit l < n/4-1 holds the complex elements k = l+1
// (ar, ai) and n/2-k (br, bi), which the split steps mix with each other and
// with nothing else; unit n/4-1 holds what they leave alone, the pair of DC
// and Nyquist (ar, ai) and the middle element n/4 (br, bi).  One pass over the
// row instead of five (split, DC, gains, split, DC), every value by the same
// operations in the same order.
__device__ __forceinline__ int unit_k(int n, int l) { return (l == n / 4 - 1) ? 0 : l + 1; }
__device__ __forceinline__ int unit_kb(int n, int l) { return (l == n / 4 - 1) ? n / 4 : n / 2 - (l + 1); }
template <class T>
__device__ __forceinline__ void split_mix(T &ar, T &ai, T &br, T &bi, T wr, T wi, T c2) {
  const T c1 = T(0.5);
  const T h1r = c1 * (ar + br), h1i = c1 * (ai - bi), h2r = -c2 * (ai + bi), h2i = c2 * (ar - br);
  ar = h1r + wr * h2r - wi * h2i;
  ai = h1i + wr * h2i + wi * h2r;
  br = h1r - wr * h2r + wi * h2i;
  bi = -h1i + wr * h2i + wi * h2r;
}
template <class T>
__device__ __forceinline__ void split_gain(T &ar, T &ai, T &br, T &bi, int n, int l, const T *trf, const T *tri,
                                           const double *hl) {
  if (l < n / 4 - 1) {
    const T g1 = T(hl[l + 2]), g2 = T(hl[n / 2 - l]);
    const T wr = trf[2 * l], wi = trf[2 * l + 1], vr = tri[2 * l], vi = tri[2 * l + 1];
    split_mix(ar, ai, br, bi, wr, wi, T(-0.5));
    ar *= g1;
    ai *= g1;
    br *= g2;
    bi *= g2;
    split_mix(ar, ai, br, bi, vr, vi, T(0.5));
  } else {
    const T g0 = T(hl[1]), gn = T(hl[n / 2 + 1]), gm = T(hl[n / 4 + 1]);
    T h1r = ar;
    ar = h1r + ai;
    ai = h1r - ai;
    ar *= g0;
    ai *= gn;
    h1r = ar;
    ar = T(0.5) * (h1r + ai);
    ai = T(0.5) * (h1r - ai);
    br *= gm;
    bi *= gm;
  }
}

// Rows per block of the row kernels: a row takes ni/4 lanes (the transform
// team: one butterfly per lane per stage), each lane holding every
// (ni/4)-th point of the row, and 1024/ni rows share a 256-lane block
// (one row when ni = 1024).
struct RowMap {
  int rpb;     // rows per block
  int g;       // this lane's row within the block
  int lane;    // this lane's index within its row
  int stride;  // lanes per row
};
__device__ __forceinline__ RowMap row_map(int ni) {
  RowMap m;
  m.stride = ni >> 2;
  m.rpb = 256 / m.stride;
  m.g = threadIdx.x / m.stride;
  m.lane = threadIdx.x - m.g * m.stride;
  return m;
}
static inline int rows_per_block(int ni) { return 1024 / ni; }
// launch of a row kernel: its WIDE form for rows of more than 256 points
#define ROWS_LAUNCH(b, name, kw, kn, g, blk, shm, s, ...)            \
  do {                                                              \
    if ((b).ni > 256) LAUNCH_AS(name, kw, g, blk, shm, s, __VA_ARGS__); \
    else LAUNCH_AS(name, kn, g, blk, shm, s, __VA_ARGS__);          \
  } while (0)

// Whether some row of this lane's synchronisation group (its wavefront when
// a row's ni/4 lanes lie in one, else its block) is to be filtered: the same
// answer in every lane of the group, which may then skip the transform's
// barriers and stages together.  Half of the rows lie outside the band.
template <bool WIDE>
__device__ __forceinline__ bool filter_any(bool active) {
  if constexpr (WIDE) return __syncthreads_or(active);
  else return __any(active);
}

// Filter one latitude row held in registers, in place: v[q] is point
// I = 1 + lane + q ni/4 of the row, lane the caller's index within its row
// (RowMap::lane), the row's ni/4 lanes being the transform team; work is ni
// values of scratch LDS of the row's own.  When ni <= 256 the team lies in
// one wavefront and the stages are separated by wavefront barriers; when
// ni > 256 by block barriers, so every lane of the block must call.  active =
// the row is in the filter band; it is untouched otherwise.  work is free
// for other use when the call returns.  The operations are those
// of the reference's realft, in its order.
template <bool WIDE, class T>
__device__ __forceinline__ void filter_row_regs(const MemberDesc &d, T (&v)[4], T *work, int J, int vgrid, bool active,
                                                int lane) {
  const int n = d.ni, nq = n >> 2, bits = d.nlogn - 1;
  const double *hl = (vgrid ? d.hl_pv : d.hl_h) + (size_t)J * (n / 2 + 2);
  if (active)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = lane + q * nq;
      work[2 * swz(brev(e >> 1, bits)) + (e & 1)] = v[q];
    }
  row_sync<WIDE>();
  four1_stages<WIDE>(work, n, lane, tw_fwd<T>(d), active);
  const int ka = unit_k(n, lane), kb = unit_kb(n, lane);
  T ar, ai, br, bi;
  if (active) {
    const int pa = 2 * swz(ka), pb = 2 * swz(kb);
    ar = work[pa];
    ai = work[pa + 1];
    br = work[pb];
    bi = work[pb + 1];
    split_gain(ar, ai, br, bi, n, lane, tr_fwd<T>(d), tr_inv<T>(d), hl);
  }
  row_sync<WIDE>();
  if (active) {
    const int pa = 2 * swz(brev(ka, bits)), pb = 2 * swz(brev(kb, bits));
    work[pa] = ar;
    work[pa + 1] = ai;
    work[pb] = br;
    work[pb + 1] = bi;
  }
  row_sync<WIDE>();
  four1_stages<WIDE>(work, n, lane, tw_inv<T>(d), active);
  if (active)
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = work[swz_val(lane + q * nq)] * T(2. / (n));
  row_sync<WIDE>();
}

// The same filter by one wavefront on `rows` rows that lie in LDS at X + r*WS
// (rows 1/64 of the NV values a lane holds of them: NV = rows*ni/64, at least
// 1); on[r] tells whether row r, row J of the grid at r = 0, is in the filter
// band (rows that are not stay as they are).  The lanes share the units of
// all rows, so that short rows fill the wavefront too, and only wavefront
// barriers separate the stages.  On entry (behind a barrier) a row that is on
// holds its points in bit-reversed order (rev_pos); on exit (behind one) the
// unscaled result, value e at swz_val(e), to be multiplied by 2/ni.
__device__ __forceinline__ int rev_pos(int e, int bits) { return 2 * swz(brev(e >> 1, bits)) + (e & 1); }
template <class T, int NV>
__device__ __forceinline__ void filter_wave(const MemberDesc &d, T *X, int WS, int rows, const int *on, int J,
                                            int vgrid, int lane) {
  const int n = d.ni, lg = d.nlogn, bits = lg - 1, S = lg - 1;
  auto stages = [&](const T *tw) {
    int s = 0;
    for (; s + 1 < S; s += 2) {
#pragma unroll
      for (int i = 0; i < (NV + 7) / 8; i++) {
        const int u = lane + 64 * i, r = u >> (lg - 3);
        if (r < rows && on[r]) four1_pair(X + r * WS, s, u & ((n >> 3) - 1), tw);
      }
      wave_sync();
    }
    if (s < S) {
#pragma unroll
      for (int i = 0; i < (NV + 3) / 4; i++) {
        const int u = lane + 64 * i, r = u >> (lg - 2);
        if (r < rows && on[r]) four1_last(X + r * WS, s, u & ((n >> 2) - 1), tw);
      }
      wave_sync();
    }
  };
  stages(tw_fwd<T>(d));
  T ar[(NV + 3) / 4], ai[(NV + 3) / 4], br[(NV + 3) / 4], bi[(NV + 3) / 4];
#pragma unroll
  for (int i = 0; i < (NV + 3) / 4; i++) {
    const int u = lane + 64 * i, r = u >> (lg - 2), l = u & ((n >> 2) - 1);
    if (r < rows && on[r]) {
      const T *x = X + r * WS;
      const int ka = unit_k(n, l), kb = unit_kb(n, l);
      const int pa = 2 * swz(ka), pb = 2 * swz(kb);
      ar[i] = x[pa];
      ai[i] = x[pa + 1];
      br[i] = x[pb];
      bi[i] = x[pb + 1];
      const double *hl = (vgrid ? d.hl_pv : d.hl_h) + (size_t)(J + r) * (n / 2 + 2);
      split_gain(ar[i], ai[i], br[i], bi[i], n, l, tr_fwd<T>(d), tr_inv<T>(d), hl);
    }
  }
  wave_sync();
#pragma unroll
  for (int i = 0; i < (NV + 3) / 4; i++) {
    const int u = lane + 64 * i, r = u >> (lg - 2), l = u & ((n >> 2) - 1);
    if (r < rows && on[r]) {
      T *x = X + r * WS;
      const int pa = 2 * swz(brev(unit_k(n, l), bits)), pb = 2 * swz(brev(unit_kb(n, l), bits));
      x[pa] = ar[i];
      x[pa + 1] = ai[i];
      x[pb] = br[i];
      x[pb + 1] = bi[i];
    }
  }
  wave_sync();
  stages(tw_inv<T>(d));
}

}  // namespace epic
