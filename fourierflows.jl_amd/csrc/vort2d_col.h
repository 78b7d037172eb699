// The single-team column kernel of the fused 2D vorticity steps and its
// launcher, shared by the ETDRK4 stages (vort2d_fused.hip) and the explicit
// steppers (vort2d_explicit.hip).
#pragma once

#include "vort2d_team3.h"

namespace ffhip {

#ifndef FF_COL_PAIR
#define FF_COL_PAIR 1  // FP32 column pass up to 1024: paired transforms (LDS has room there)
#endif
template <typename R, int N>
constexpr bool col_pair() {
  return sizeof(R) == 4 && N <= 1024 && FF_COL_PAIR;
}

#ifndef FF_COL_WAVES
#define FF_COL_WAVES 1  // minimum FP32 waves per SIMD the column pass is compiled for
#endif
#ifndef FF_COL_WAVES_F64
#define FF_COL_WAVES_F64 1
#endif

// Columns per workgroup: kCBK, but one for FP64 4096-point columns (a
// column's buffer and twiddle table take 135 KB of LDS).
template <typename R, int NY>
constexpr int col_cbk() {
  return sizeof(R) == 8 && NY == 4096 ? 1 : kCBK;
}

// STAGE 0: y-inverse of U only.  STAGE 1..4: ETDRK4 stages; 5: explicit steppers.  col_cbk columns
// per workgroup; the workgroups of one 4-column tile run on the same XCD.
template <typename R, int NY, int P, int STAGE>
__global__ void __launch_bounds__((col_cbk<R, NY>() * (NY / P)), (sizeof(R) == 4 ? FF_COL_WAVES : FF_COL_WAVES_F64))
    k_vcol(VortGeom g, VortColArgs a) {
  extern __shared__ unsigned char vsm[];
  constexpr int CB = col_cbk<R, NY>();
  int tx, sub;
  xcd_split(blockIdx.x, kVCB / CB, &tx, &sub);
  if (tx >= g.TX) return;  // grid is rounded up to whole XCD groups
  const int t = threadIdx.x;
  const int cc = t % CB;
  constexpr int SL = team_slice(TeamSched<NY, P>::LDS, sizeof(cplx<R>), CB);
  constexpr bool pair = col_pair<R, NY>();  // second buffers after the first, then the table
  cplx<R>* base = reinterpret_cast<cplx<R>*>(vsm);
  const cplx<R>* tw = team_tw_load<NY, P, R>(base + (pair ? 2 : 1) * CB * SL, a.tw);
  vcol_body<R, NY, P, STAGE, pair>(g, a, tx, sub * CB + cc, t / CB, base + cc * SL, tw, true,
                                   pair ? base + (CB + cc) * SL : nullptr);
}

template <typename R, int N>
static size_t col_lds() {
  constexpr int CB = col_cbk<R, N>();
  constexpr size_t sl = team_slice(TeamSched<N, vcol_pts<R, N>()>::LDS, sizeof(cplx<R>), CB);
  return ((col_pair<R, N>() ? 2 : 1) * CB * sl + tw_slots<N, vcol_pts<R, N>()>()) * sizeof(cplx<R>);
}

static const char* const kColNames[6] = {"vort_col_stage0", "vort_col_stage1", "vort_col_stage2",
                                         "vort_col_stage3", "vort_col_stage4", "vort_col_explicit"};

template <typename R, int N, int STAGE>
static int launch_col_team(const VortGeom& g, const VortColArgs& a, hipStream_t st) {
  constexpr int P = vcol_pts<R, N>();
  const size_t sh = col_lds<R, N>();
  auto kern = k_vcol<R, N, P, STAGE>;
  static bool attr_set = false;
  if (!attr_set) {
    FF_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sh));
    attr_set = true;
  }
  const int groups = (g.TX + kXCD - 1) / kXCD * kXCD;
  constexpr int CB = col_cbk<R, N>();
  prof_launch(kColNames[STAGE], col_bytes<R>(g, STAGE, a.do_inverse), kern,
              dim3(groups * (kVCB / CB)), dim3(CB * (N / P)), sh, st, g, a);
  FF_LAUNCHED("k_vcol");
  return FFHIP_OK;
}

template <typename R, int N, int STAGE, int P, int C, int W = 1>
static int launch_colt(const VortGeom& g, const VortColArgs& a, hipStream_t st) {
  constexpr size_t sh = vcolt_lds<R, N, P, C>();
  auto kern = k_vcolt<R, N, P, STAGE, C, W>;
  static bool attr_set = false;
  if (!attr_set) {
    FF_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sh));
    attr_set = true;
  }
  const int groups = (g.TX + kXCD - 1) / kXCD * kXCD;
  prof_launch(kColNames[STAGE], col_bytes<R>(g, STAGE, a.do_inverse), kern, dim3(groups * (kVCB / C)),
              dim3(3 * C * (N / P)), sh, st, g, a);
  FF_LAUNCHED("k_vcolt");
  return FFHIP_OK;
}

// Three teams per column (vort2d_team3.h) up to 256 points and, up to a number
// of columns, at 512 and 1024; the single-team kernel beyond.
// Stage 2 on an n x n grid, single team -> three teams, MI355X: FP64 64^2 7.6
// -> 3.5 us, 128^2 9.0 -> 4.2, 256^2 17.1 -> 5.1, 512^2 17.2 -> 7.4; FP32 64^2
// 6.2 -> 3.5, 128^2 7.0 -> 4.1, 256^2 12.0 -> 4.7, 512^2 7.8 -> 6.2, 1024^2
// 14.8 -> 12.5.  With 683 columns (nx = 2048) FP32 loses at 512 (9.5 -> 9.7)
// and 1024 (19.0 -> 22.7), FP64 at 1024 already with 341 (stage 4: 25.6 ->
// 32 us, its operands spill).  FP64 512 points, single team -> three teams:
// stage 1 with 171 tiles of columns (nx = 2048) 21.9 -> 16.0, 257 24.9 -> 23.0,
// 342 (nx = 4096) 27.1 -> 27.1 and stage 2 28.6 -> 25.4; stage 4, the one with
// most operands, 171 22.3 -> 19.4, 235 23.7 -> 23.3, 257 25.0 -> 26.5, 342 27.1
// -> 31.3.  Up to 256 points three teams win at every width up to 4096 (FP64
// 256 x 4096 23.2 -> 12.3).  With many short columns two per workgroup use
// the lines better (128-point FP32, nx = 4096: 7.0 -> 5.9 us).
template <typename R, int N, int STAGE>
static int launch_col(const VortGeom& g, const VortColArgs& a, hipStream_t st) {
  constexpr bool f32 = sizeof(R) == 4;
  if constexpr (N <= 128) {
    return g.TX <= 96 ? launch_colt<R, N, STAGE, 4, 1>(g, a, st) : launch_colt<R, N, STAGE, 4, 2>(g, a, st);
  } else if constexpr (N == 256) {
    return g.TX <= 96 ? launch_colt<R, N, STAGE, 4, 1>(g, a, st) : launch_colt<R, N, STAGE, 8, 2>(g, a, st);
  } else if constexpr (N == 512 && !f32) {
    if (g.TX <= (STAGE == 4 ? 240 : 344)) return launch_colt<R, N, STAGE, 8, 1>(g, a, st);
    return launch_col_team<R, N, STAGE>(g, a, st);
  } else {
    if constexpr (N == 512) {
      if (g.TX <= 88) return launch_colt<R, N, STAGE, 8, 1>(g, a, st);
    } else if constexpr (N == 1024) {
      if (g.TX <= (f32 ? 88 : 44)) return launch_colt<R, N, STAGE, 16, 1, 2>(g, a, st);
    }
    return launch_col_team<R, N, STAGE>(g, a, st);
  }
}

}  // namespace ffhip
