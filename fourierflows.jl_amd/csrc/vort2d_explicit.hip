// The explicit steppers (ForwardEuler, RK4, AB3, LSRK54 and their filtered
// forms, src/timesteppers.jl:98-414, 588-666) of built-in 2D vorticity on the
// fused row and column passes: two launches per stage, where the plan-based
// path needs 15 to 17 (four transforms of two passes each way, the products
// and the updates).  The stage updates run inside the column kernel
// (xstage_point); U, RHS_1..3 and L stay in the kept band's blocked layout
// between stages.
//
// Measured on MI355X, FilteredRK4 at 512^2 FP32: 206 us per step on the
// plan-based path, 51 us here (row passes 4.8 us, column stages 6.2 us, of which
// 0.8 and 0.6 are VALU issue: latency, as in the ETDRK4 steps).
#include "vort2d_col.h"

namespace ffhip {

// Gather the state, L, the filter and AB3's history into the blocked layout
template <typename R>
__global__ void k_ximport(const cplx<R>* __restrict__ sol, cplx<R>* __restrict__ U, const double* __restrict__ L,
                          double* __restrict__ XL, const double* __restrict__ F, double* __restrict__ XF,
                          const cplx<R>* __restrict__ m1, cplx<R>* __restrict__ R1, const cplx<R>* __restrict__ m2,
                          cplx<R>* __restrict__ R2, VortGeom g) {
  const int64_t total = (int64_t)g.TX * g.KY * kVCB;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(idx % kVCB);
    const int64_t rest = idx / kVCB;
    const int ky = (int)(rest % g.KY);
    const int ix = (int)(rest / g.KY) * kVCB + c;
    const bool live = ix < g.KX;
    const int64_t src = (int64_t)v_iy(ky, g) * g.nkr + ix;
    U[idx] = live ? sol[src] : mkc<R>(0, 0);
    XL[idx] = live ? L[src] : 0.0;
    if (F) XF[idx] = live ? F[src] : 0.0;
    if (m1) {
      R1[idx] = live ? m1[src] : mkc<R>(0, 0);
      R2[idx] = live ? m2[src] : mkc<R>(0, 0);
    }
  }
}

// Scatter the kept band back; outside it N is zero and each mode takes its
// nsteps steps here, rounding where the plan-based path's arrays do (zeros
// stay: all of them where L is finite).
template <typename R>
__global__ void k_xexport(cplx<R>* __restrict__ sol, const cplx<R>* __restrict__ U, const double* __restrict__ L,
                          const double* __restrict__ F, cplx<R>* __restrict__ m1, const cplx<R>* __restrict__ R1,
                          cplx<R>* __restrict__ m2, const cplx<R>* __restrict__ R2, int kind, double h, double h2,
                          int64_t nsteps, int64_t step0, bool zeros_stay, VortGeom g) {
  const int64_t total = (int64_t)g.ny * g.nkr;
  const cplx<R> zero = mkc<R>(0, 0);
  const bool f32 = sizeof(R) == 4;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int ix = (int)(idx % g.nkr);
    const int iy = (int)(idx / g.nkr);
    if (ix < g.KX && (iy < g.ylo || iy > g.yhi)) {
      const int64_t b = ((int64_t)(ix / kVCB) * g.KY + v_ky(iy, g)) * kVCB + ix % kVCB;
      sol[idx] = U[b];
      if (m1) {
        m1[idx] = R1[b];
        m2[idx] = R2[b];
      }
      continue;
    }
    cplx<R> u = sol[idx];
    cplx<R> r1 = m1 ? m1[idx] : zero, r2 = m1 ? m2[idx] : zero;
    const double l = L[idx];
    if (!zeros_stay || u.x != R(0) || u.y != R(0) || r1.x != R(0) || r1.y != R(0) || r2.x != R(0) || r2.y != R(0)) {
      const double f = F ? F[idx] : 1.0;
      for (int64_t k = 0; k < nsteps; ++k) {
        if (kind == 0) {
          u = xeuler_end<R>(u, zero, l, h, f);
          continue;
        }
        if (kind == 1) {
          const cplx<R> r = xrhs<R>(l, u, zero);
          u = step0 + k < 3 ? xadd<R>(u, r, h) : xab3_end<R>(u, r, r1, r2, h);
          r2 = r1;
          r1 = r;
        } else if (kind == 2) {
          cplx<R> s2 = zero;
          for (int i = 0; i < 5; ++i) {
            // the coefficients in the state's type, as the stages on the band take them
            s2 = xlsrk_s2<R>(s2, xrhs<R>(l, u, zero), f32 ? (double)(float)kLsrkA[i] : kLsrkA[i], h);
            u = xadd<R>(u, s2, f32 ? (double)(float)kLsrkB[i] : kLsrkB[i]);
          }
        } else {
          const cplx<R> q1 = xrhs<R>(l, u, zero);
          const cplx<R> q2 = xrhs<R>(l, xadd<R>(u, q1, h2), zero);
          const cplx<R> q3 = xrhs<R>(l, xadd<R>(u, q2, h2), zero);
          const cplx<R> q4 = xrhs<R>(l, xadd<R>(u, q3, h), zero);
          u = xrk4_end<R>(u, q1, q2, q3, q4, h / 6);
        }
        if (F) u = xscale<R>(u, f);
      }
      sol[idx] = u;
      if (m1) {
        m1[idx] = r1;
        m2[idx] = r2;
      }
    }
  }
}

template <typename R>
static int xcol(const VortGeom& g, const VortColArgs& a, hipStream_t st) {
  switch (g.ny) {
    case 64: return launch_col<R, 64, kVExplicit>(g, a, st);
    case 128: return launch_col<R, 128, kVExplicit>(g, a, st);
    case 256: return launch_col<R, 256, kVExplicit>(g, a, st);
    case 512: return launch_col<R, 512, kVExplicit>(g, a, st);
    case 1024: return launch_col<R, 1024, kVExplicit>(g, a, st);
    case 2048: return launch_col<R, 2048, kVExplicit>(g, a, st);
    case 4096: return launch_col<R, 4096, kVExplicit>(g, a, st);
    default: return fail(FFHIP_ERR_UNSUPPORTED, "fused column kernel: ny = %d", g.ny);
  }
}

int vort_col_explicit(int prec, const VortGeom& g, const VortColArgs& a, hipStream_t st) {
  return prec == FFHIP_F32 ? xcol<float>(g, a, st) : xcol<double>(g, a, st);
}

template <typename R>
static int xrun(ffhip_op* op, VortState* s, ffhip_rk4* ts, int kind, void* sol, double dt, int64_t nsteps, int64_t step0, void* m1,
                void* m2, hipStream_t st) {
  const VortGeom& g = s->g;
  const int prec = op->prec;
  const int64_t n = (int64_t)g.TX * g.KY * kVCB;
  const double h2 = prec == FFHIP_F32 ? (double)((float)dt / 2.0f) : dt / 2;
  const double* F = reinterpret_cast<const double*>(ts->filter);
  const bool ab3 = kind == 1;
  cplx<R>* m1p = ab3 ? reinterpret_cast<cplx<R>*>(m1) : nullptr;
  cplx<R>* m2p = ab3 ? reinterpret_cast<cplx<R>*>(m2) : nullptr;
  hipLaunchKernelGGL((k_ximport<R>), dim3(blocks_for(n, 256, 4096)), dim3(256), 0, st,
                     reinterpret_cast<const cplx<R>*>(sol), reinterpret_cast<cplx<R>*>(s->U),
                     reinterpret_cast<const double*>(ts->L), reinterpret_cast<double*>(s->XL), F,
                     reinterpret_cast<double*>(s->XF), m1p, reinterpret_cast<cplx<R>*>(s->N1), m2p,
                     reinterpret_cast<cplx<R>*>(s->N2), g);
  FF_LAUNCHED("k_ximport");
  VortColArgs ca{};
  ca.O0 = s->O[0];
  ca.O1 = s->O[1];
  ca.I0 = s->I[0];
  ca.I1 = s->I[1];
  ca.I2 = s->I[2];
  ca.U = s->U;
  ca.N1 = s->N1;
  ca.N2 = s->N2;
  ca.A = s->A;
  ca.tw = s->twy;
  ca.do_inverse = 1;
  ca.L = reinterpret_cast<const double*>(s->XL);
  VortRowArgs ra;
  ra.I0 = s->I[0];
  ra.I1 = s->I[1];
  ra.I2 = s->I[2];
  ra.O0 = s->O[0];
  ra.O1 = s->O[1];
  ra.tw = s->twx;
  ra.F = nullptr;
  FF_TRY(vort_col_any(prec, 0, s, ca, st));
  const double* fl = F ? reinterpret_cast<const double*>(s->XF) : nullptr;
  // one stage: row pass, then the column pass with the stage update; `end`
  // marks the stage that completes a step (the filter acts there), and the
  // last one of the run skips its inverse transforms
  auto stage = [&](int xkind, double c0, double c1, double c2, bool end, bool last) -> int {
    FF_TRY(vort_row_any(prec, s, ra, st));
    ca.kind = xkind;
    ca.c0 = c0;
    ca.c1 = c1;
    ca.c2 = c2;
    ca.Fl = end ? fl : nullptr;
    ca.do_inverse = !(end && last);
    return vort_col_any(prec, kVExplicit, s, ca, st);
  };
  const bool f32 = prec == FFHIP_F32;
  for (int64_t k = 0; k < nsteps; ++k) {
    const bool last = k + 1 == nsteps;
    if (kind == 0) {
      FF_TRY(stage(kXEuler, dt, 0, 0, true, last));
    } else if (ab3) {
      FF_TRY(stage(step0 + k < 3 ? kXAB3start : kXAB3, dt, 0, 0, true, last));
      std::swap(ca.N1, ca.N2);  // the new RHS is RHS_-1 of the next step
    } else if (kind == 2) {
      for (int i = 0; i < 5; ++i)
        FF_TRY(stage(kXLSRK, f32 ? (double)(float)kLsrkA[i] : kLsrkA[i], f32 ? (double)(float)kLsrkB[i] : kLsrkB[i], dt,
                     i == 4, last));
    } else {
      for (int i = 0; i < 4; ++i) FF_TRY(stage(kXRK4a + i, h2, dt, dt / 6, i == 3, last));
    }
  }
  const int64_t total = (int64_t)g.ny * g.nkr;
  hipLaunchKernelGGL((k_xexport<R>), dim3(blocks_for(total, 256, 4096)), dim3(256), 0, st,
                     reinterpret_cast<cplx<R>*>(sol), reinterpret_cast<const cplx<R>*>(s->U),
                     reinterpret_cast<const double*>(ts->L), F, m1p, reinterpret_cast<const cplx<R>*>(ca.N1), m2p,
                     reinterpret_cast<const cplx<R>*>(ca.N2), kind, dt, h2, nsteps, step0,
                     ts->L_finite, g);
  FF_LAUNCHED("k_xexport");
  return FFHIP_OK;
}

int fused_explicit_run(ffhip_op* op, ffhip_rk4* ts, int kind, void* sol, double dt, int64_t nsteps, int64_t step0,
                       void* m1, void* m2, bool* done, hipStream_t st) {
  VortState* s = ts->cplx_coef ? nullptr : vort_state(op, st);
  if (!s || (!s->mixx && !vort_row_ok(op->prec, s->g))) return FFHIP_OK;
  const size_t bytes = (size_t)s->g.TX * s->g.KY * kVCB * sizeof(double);
  // a capture cannot allocate: the plan-based path takes its first run
  if ((!s->XL || (ts->filter && !s->XF)) && vort_capturing(st)) return FFHIP_OK;
  if ((!s->XL && dev_alloc(&s->XL, bytes) != FFHIP_OK) ||
      (ts->filter && !s->XF && dev_alloc(&s->XF, bytes) != FFHIP_OK)) {
    clear_error();  // no room for the blocked copies: the plan-based path runs
    return FFHIP_OK;
  }
  *done = true;
  return op->prec == FFHIP_F32 ? xrun<float>(op, s, ts, kind, sol, dt, nsteps, step0, m1, m2, st)
                               : xrun<double>(op, s, ts, kind, sol, dt, nsteps, step0, m1, m2, st);
}

}  // namespace ffhip
