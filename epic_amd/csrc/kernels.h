// kernels.h -- host-side launchers of the engine's HIP kernels.
// Every launcher covers the members [mb, mb+nm) of one bucket (same ni,nj,nk)
// on stream s.  Field selectors name a 3-D array of the MemberDesc.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "dev_common.h"

namespace epic {

// Optional per-launch timing: when enabled, every launch is bracketed by HIP
// events on its stream and the durations are aggregated per kernel name.
void prof_begin(hipStream_t s, const char *name);
void prof_end(hipStream_t s);
extern bool g_prof_on;
#define LAUNCH(k, g, b, shm, s, ...) LAUNCH_AS(#k, k, g, b, shm, s, __VA_ARGS__)
// the same under a given profile name (for a kernel whose template arguments
// hold commas, which is passed in parentheses)
#define LAUNCH_AS(name, k, g, b, shm, s, ...)            \
  do {                                                   \
    if (::epic::g_prof_on) ::epic::prof_begin(s, name);  \
    hipLaunchKernelGGL(k, g, b, shm, s, __VA_ARGS__);    \
    if (::epic::g_prof_on) ::epic::prof_end(s);          \
  } while (0)

// Up to four fields processed by one launch of a batched kernel, each with
// its kind (0 U, 1 V, 2 HDRY, 3 THETA); blockIdx.z = field index * members
// + member, and field i uses scratch copy copy0 + i.
struct FieldSet {
  int n;
  int f[4], kind[4];
  int copy0;
};

// Launch shapes a bucket can be tuned over (epic_engine_autotune); 0 takes
// the built-in choice.  None of them changes a result: every cell is formed
// by the same operations whatever the tile.
enum Knob { KN_COLS_P2ETC, KN_COLS_GZ3, KN_COLS_CALCW, KN_COLS_HSUV, KN_ROWS_ZHV, KN_ROWS_MER, KN_ROWS_D2, KN_COUNT };
// A column-tile knob holds the columns per block C and, from 1000 up, the
// threads asked for: v = C (256 threads), v = 1000 n + C (256 n threads,
// n = 2 or 4), or v = 10000 + C (one for each of the column's `levels`).  The
// Akima column pass's block has these threads; set_p2etc, gz3 and calc_w give
// a thread 2, 4 or 8 levels, the fewest that such a block covers the column
// with (8 where it cannot), and take the threads that this needs (col_shape).
static inline int knob_cols(int v) { return v % 1000; }
static inline int knob_threads(int v, int levels) {
  return v >= 10000 ? (v % 1000) * levels : v >= 1000 ? (v / 1000) * 256 : 256;
}

struct Bucket {
  const MemberDesc *D;  // device array of descriptors
  int mb, nm;           // first member, member count
  int ni, nj, nk;
  int mixed;            // FP32 tendencies and horizontal arithmetic
  int knob[KN_COUNT];   // columns per column tile / rows per zonal-mean block
  // some member is a gas giant (gz_from_u), Held-Suarez (boundary-layer
  // drag), or has Rayleigh drag: launches none of the members needs are
  // left out (their kernels would return at once for every member)
  int any_gas, any_hs, any_ray;
  // hyperviscosity passes of the member that needs the most (hv_passes)
  int hv_passes;
  // advection schemes some member's field takes: bit 0 Hsu-Konor-Arakawa,
  // bit 1 Akima (the launches of a scheme no field takes are left out)
  int adv_schemes;
};

// The shape of a column-tile kernel (set_p2etc, gz3, calc_w): columns, levels
// per lane, threads
struct ColShape {
  int C, KC, nt;
};
inline ColShape col_shape(const Bucket &b, int knob) {
  const int lev = b.nk;
  ColShape s{64, 2, 0};
  if (knob) {
    s.C = knob_cols(knob);
    const int groups = std::max(1, knob_threads(knob, lev + 1) / s.C);
    while (s.KC < 8 && groups * s.KC < lev) s.KC *= 2;
  } else {
    // More levels a lane read and form fewer around them again, but leave
    // fewer wavefronts: the most that leave 8192 (8 levels) or 2048 (4) of
    // them.  Steps with 2, 4 and 8 levels: 64x32x10 170, 181, 208 us;
    // 256x128x20 441, 442, 469; 23 members of 128x51x13 955, 952, 981; 64 mixed
    // ones of 128x64x16 3510, 3414, 3310; mixed 512x256x32 1786, 1786, 1759.
    const size_t tiles = ((size_t)(b.nj + 1) * (b.ni + 2) + 63) / 64 * b.nm;
    s.KC = tiles * ((lev + 7) / 8) >= 8192 ? 8 : tiles * ((lev + 3) / 4) >= 2048 ? 4 : 2;
  }
  // (any depth: 8 columns take up to 1024 levels)
  while (s.KC < 8 && (lev + s.KC - 1) / s.KC * s.C > 1024) s.KC *= 2;
  while (s.C > 1 && (lev + s.KC - 1) / s.KC * s.C > 1024) s.C /= 2;
  s.nt = s.C * ((lev + s.KC - 1) / s.KC);
  return s;
}
// its LDS: one column of nk+1 values for each of its columns
inline size_t col_lds(const Bucket &b, int C) { return sizeof(double) * C * (b.nk + 1); }
// the Akima column pass's LDS (of FP64 values): four columns of nk+2 values each
inline size_t ak_col_lds(const Bucket &b, int C) { return sizeof(double) * 4 * C * (b.nk + 2); }

// the Bucket::adv_schemes bits of one member
inline int adv_schemes(const MemberDesc &d) {
  int s = 0;
  for (int f = 0; f < 3; f++) s |= d.adv_akima[f] ? 2 : 1;
  return s;
}

// ---- diagnostics (k_diag.hip)
void L_fill(hipStream_t s, const Bucket &b, int fld, double v);
void L_set_p2etc(hipStream_t s, const Bucket &b, int update_theta);
void L_richardson(hipStream_t s, const Bucket &b);
void L_gz_from_u(hipStream_t s, const Bucket &b);
void L_gz3(hipStream_t s, const Bucket &b);
void L_dzdt3(hipStream_t s, const Bucket &b);
void L_heating(hipStream_t s, const Bucket &b, int adjust, bool in_thermo);
void L_calc_w(hipStream_t s, const Bucket &b, int with_source);
void L_divergence(hipStream_t s, const Bucket &b, int uu, int vv, int dst, int k0, int k1);
// store_diag (PV3 and DIV_UV3 of U, V on K = 0..nk) in one launch; rotate:
// also rotate the time planes and advance itime (the step's last action)
void L_store_diag(hipStream_t s, const Bucket &b, int rotate);
// store_pgrad_vars' per-cell values after the FULL set_p2etc
void L_thermo(hipStream_t s, const Bucket &b);

// ---- zonal filter (k_filter.hip)
// the 3-D filter with the PCHIP profile removal, on every field of the set
void L_filter3(hipStream_t s, const Bucket &b, const FieldSet &fs);

// ---- momentum (k_dyn.hip)
void L_uv_core(hipStream_t s, const Bucket &b);
void L_uv_drag(hipStream_t s, const Bucket &b);
void L_pgrad(hipStream_t s, const Bucket &b);
void L_divdamp(hipStream_t s, const Bucket &b);
// the Adams-Bashforth update; where ab_dzdt3_fused, DZDT3 too
bool ab_dzdt3_fused(const Bucket &b);
void L_ab(hipStream_t s, const Bucket &b);
void L_gz_mono(hipStream_t s, const Bucket &b);
void L_gz_filtercopy(hipStream_t s, const Bucket &b);
// hyperviscosity on every field of the set (at most two: the meridional
// part keeps its del^4 result in scratch copy i of sB)
void L_merid_hv(hipStream_t s, const Bucket &b, const FieldSet &fs);
void L_zonal_hv(hipStream_t s, const Bucket &b, const FieldSet &fs);
// hyperviscosity of hdry and theta (before the advection) and of u and v;
// hv_fused: as one launch each, through sD's copies 1 and 2
bool hv_fused(const Bucket &b);
void L_hv_hth(hipStream_t s, const Bucket &b);
void L_hv_uv(hipStream_t s, const Bucket &b);

// ---- mixed-precision momentum kernels (k_mixed.hip)
void LM_uv_drag(hipStream_t s, const Bucket &b);
void LM_divdamp_apply(hipStream_t s, const Bucket &b);

// ---- advection (k_adv.hip)
void L_advection(hipStream_t s, const Bucket &b);

}  // namespace epic
