// Built-in operator object shared by the generic and fused paths.
#pragma once

#include <cstdint>

#include "plan.h"
#include "stepper.h"

struct ffhip_op {
  int kind = 0;
  int prec = FFHIP_F64;
  int ndim = 2;
  int64_t n[3] = {1, 1, 1};   // nx, ny, nz
  double box[3] = {1, 1, 1};  // Lx, Ly, Lz
  double af = 1.0 / 3.0;      // aliased_fraction
  double params[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int nparams = 0;
  int64_t nkr = 1;
  int64_t spec_count = 0, phys_count = 0;
  int64_t lo[3] = {1, 1, 1}, hi[3] = {0, 0, 0};  // 1-based aliased ranges on the rfft layout
  ffhip_plan* plan = nullptr;
  void* spec[3] = {nullptr, nullptr, nullptr};
  void* phys[4] = {nullptr, nullptr, nullptr, nullptr};
  void* tables = nullptr;  // tracer: sin/cos of the grid coordinates (FP64)
  void* fused = nullptr;   // fused implementation state (power-of-two vorticity grids)
  void* mixed = nullptr;   // the same on other grids (mixed-radix passes), made at the first run
  bool no_mixed = false;   // that state is not wanted, not possible or found no memory
  bool no_modes = false;   // tracer: transforms also where the mode stencil would do
  void* flags = nullptr;   // tracer: three ints of the mode stencil (tracer_modes.hip)
  void* fused3 = nullptr;  // fused RK4 state of the tracer (power-of-two 3D grids)
};

namespace ffhip {

int op_calcN(ffhip_op* op, void* N, const void* sol, hipStream_t st);
// fused path (vort2d_fused.hip): create sets op->fused when the grid qualifies
int fused_create(ffhip_op* op);
void fused_destroy(ffhip_op* op);
// (*done stays false, and nothing has run, where the fused passes do not take the grid)
int fused_etdrk4_run(ffhip_op* op, ffhip_etdrk4* ts, void* sol, int64_t nsteps, bool* done, hipStream_t st);
// explicit steppers on the fused passes (vort2d_explicit.hip).  kind: 0 ForwardEuler, 1 AB3, 2 LSRK54, 3 RK4.
// *done stays false (and nothing has run) where the fused passes do not take the operator.
int fused_explicit_run(ffhip_op* op, ffhip_rk4* ts, int kind, void* sol, double dt, int64_t nsteps, int64_t step0,
                       void* m1, void* m2, bool* done, hipStream_t st);
// LSRK54 coefficients (src/timesteppers.jl:330-345), Carpenter & Kennedy (1994)
inline constexpr double kLsrkA[5] = {0.0, -567301805773.0 / 1357537059087.0, -2404267990393.0 / 2016746695238.0,
                                     -3550918686646.0 / 2091501179385.0, -1275806237668.0 / 842570457699.0};
inline constexpr double kLsrkB[5] = {1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0,
                                     1720146321549.0 / 2090206949498.0, 3134564353537.0 / 4481467310338.0,
                                     2277821191437.0 / 14882151754819.0};
// fused tracer RK4 (tracer3d_fused.hip)
int tracer_fused_create(ffhip_op* op);
void tracer_fused_destroy(ffhip_op* op);
int tracer_fused_rk4_run(ffhip_op* op, ffhip_rk4* ts, void* sol, double dt, int64_t nsteps, hipStream_t st);
int tracer_fused_rk4_adjoint(ffhip_op* op, ffhip_rk4* ts, void* lam, double dt, int64_t nsteps, hipStream_t st);
// the tracer as a stencil over modes (tracer_modes.hip); *done stays false, and
// nothing has run, where the box or the band does not allow it
int tracer_modes_calcN(ffhip_op* op, void* N, const void* sol, bool* done, hipStream_t st);
int tracer_modes_rk4(ffhip_op* op, const ffhip_rk4* ts, void* sol, double dt, int64_t nsteps, bool* done,
                     hipStream_t st);
// discrete adjoint (vort2d_adjoint.hip)
int fused_forward_ckpt(ffhip_op* op, ffhip_etdrk4* ts, const void* sol0, void* solT, int64_t nsteps,
                       int64_t ncheck, hipStream_t st);
int fused_adjoint(ffhip_op* op, ffhip_etdrk4* ts, const void* lamT, void* lam0, int64_t nsteps, int64_t ncheck,
                  hipStream_t st);
int64_t fused_checkpoint_id(const ffhip_op* op);

}  // namespace ffhip
