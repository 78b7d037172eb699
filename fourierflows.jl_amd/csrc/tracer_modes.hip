// The passive tracer in the ABC flow as a stencil over Fourier modes.
//
// On a box whose lengths are multiples of 2 pi each velocity component is two
// pairs of Fourier modes (wavenumber index q = L / 2 pi along one axis), so
// (u c)^ needs no transform: with p = exp(i x0)
//   (sin x c)^_k = (p c_{k-q} - conj(p) c_{k+q}) / 2i
//   (cos x c)^_k = (p c_{k-q} + conj(p) c_{k+q}) / 2
// and N = -i (kx U + l V + m W) reads six neighbours of a mode.  The grid's
// products give the same N to rounding as long as no product of kept modes
// aliases back to a kept one (2 kmax + q < n on every axis).  What the c2r
// ignores is left out here as well: modes outside the kept band, and the part
// of the kx = 0 plane that is not Hermitian, which also supplies the modes of
// negative kx.
//
// A mode that is infinite or NaN makes every grid value NaN and with them N on
// the whole kept band.  The stencil alone would hand it to the neighbours only,
// so the passes note one they read, and the last launch fills the band.
//
// An RK4 stage is one kernel over the kept band: it reads the stage state with
// its neighbours (from cache), the state and L, and writes RHS and the next
// stage state, so memory bounds it: 256^3 FP32 (2.5 M kept modes) moves 80 to
// 140 MB in 20 to 27 us, 4 to 5 TB/s (192^3 FP64: 13 to 19 us).  With
// transforms a stage was four kernels and 228 us.
// FP64 stage arithmetic and the state type at every store as in pointwise.hip.
#include <cmath>
#include <cstdlib>

#include "ops.h"
#include "prof.h"

namespace ffhip {

constexpr int kTmThreads = 256;
constexpr int kTmPlanes = 4;  // consecutive m of a thread (256^3 FP32 a step: 1 111 us, 2 109, 4 109, 8 117; 192^3 FP64: 97, 72, 71, 85)

struct TmGeom {
  int nkr, ny, nz;         // native layout [nz][ny][nkr]
  int KX, KY, KZ;          // kept modes, packed layout [KZ][KY][KX]
  int lmin, lmax, mmin, mmax;
  int q[3];
  int slow;                // columns kx <= q (they read the kx = 0 plane or beyond)
  int tfast, tslow;        // workgroups of a group of planes
  int per_xcd, nblk;
  float inv_fast, inv_slow;
  double dk, dl, dm;
  double p[3][2];          // (B, C, A) / 2 exp(i x0)
};

struct TmArgs {
  const void* x;  // stage state
  void* sol;
  void* out;      // next stage state, or N (stage 0)
  void* R[3];
  const double* L;
  const double* F;  // filter or null
  double h, h6;
  int* bad;   // a mode that is not finite: [0] in the run, [1] in stage 1's state, [2] in calcN's
  int first;  // stage 1 of a run
};

// a field of modes by signed wavenumbers: rows of ny_, planes of nz_ (native: ny, nz; packed: KY, KZ)
template <typename R>
struct TmField {
  const cplx<R>* p;
  int nx_, ny_, nz_;
  __device__ __forceinline__ uint32_t at(int kx, int l, int m) const {
    return (uint32_t)(((m + (m < 0 ? nz_ : 0)) * ny_ + l + (l < 0 ? ny_ : 0)) * nx_ + kx);
  }
  // zero outside the kept band
  __device__ __forceinline__ cplx<R> get(const TmGeom& g, int kx, int l, int m) const {
    if (kx >= g.KX || l < g.lmin || l > g.lmax || m < g.mmin || m > g.mmax) return mkc<R>(0, 0);
    return p[at(kx, l, m)];
  }
  // any kx: the Hermitian part on kx = 0 and conjugates below
  __device__ __forceinline__ cplx<R> get_any(const TmGeom& g, int kx, int l, int m) const {
    const bool neg = kx < 0;
    cplx<R> a = neg ? get(g, -kx, -l, -m) : get(g, kx, l, m);
    if (kx == 0) {
      const cplx<R> b = get(g, 0, -l, -m);
      a = mkc<R>(R(0.5) * (a.x + b.x), l == 0 && m == 0 ? R(0) : R(0.5) * (a.y - b.y));  // the mean is real
    }
    return neg ? cconj<R>(a) : a;
  }
};

// (a, b) = (p z_{k-q}, conj(p) z_{k+q}), p = A / 2 exp(i x0): *c = a + b = (A cos x c)^_k, *s = (a - b) / i =
// (A sin x c)^_k.  In FP64 for either state type: the velocity's coefficients are FP64 as the grid's are, N is
// rounded once, which costs FP32 little beside the memory (256^3: 102.4 -> 103.5 us a step; error of N 6.7e-8 -> 2.5e-8).
template <typename R>
__device__ __forceinline__ void tm_pair(const double* p, cplx<R> zm, cplx<R> zp, double2* c, double2* s) {
  const double ax = p[0] * (double)zm.x - p[1] * (double)zm.y, ay = p[0] * (double)zm.y + p[1] * (double)zm.x;
  const double bx = p[0] * (double)zp.x + p[1] * (double)zp.y, by = p[0] * (double)zp.y - p[1] * (double)zp.x;
  *c = make_double2(ax + bx, ay + by);
  *s = make_double2(ay - by, bx - ax);
}

template <typename R, bool SLOW>
__device__ __forceinline__ cplx<R> tm_N(const TmGeom& g, const TmField<R>& f, int kx, int l, int m) {
  auto get = [&](int a, int b, int c) { return SLOW ? f.get_any(g, a, b, c) : f.get(g, a, b, c); };
  double2 cx, sx, cy, sy, cz, sz;
  tm_pair<R>(g.p[0], get(kx - g.q[0], l, m), get(kx + g.q[0], l, m), &cx, &sx);
  tm_pair<R>(g.p[1], get(kx, l - g.q[1], m), get(kx, l + g.q[1], m), &cy, &sy);
  tm_pair<R>(g.p[2], get(kx, l, m - g.q[2]), get(kx, l, m + g.q[2]), &cz, &sz);
  const double k = g.dk * (double)kx, ll = g.dl * (double)l, mm = g.dm * (double)m;
  const double sr = k * (sz.x + cy.x) + ll * (sx.x + cz.x) + mm * (sy.x + cx.x);
  const double si = k * (sz.y + cy.y) + ll * (sx.y + cz.y) + mm * (sy.y + cx.y);
  return mkc<R>((R)si, (R)-sr);  // -i (kx U + l V + m W)
}

// What a mode's update reads, and its update.  STAGE 0: N of x to out (both
// native); 1..4: the RK4 stages.  x is native in stages 0 and 1, packed after.
template <typename R>
struct TmVal {
  cplx<R> n, u, x, r1, r2, r3;
  double L, F;
};
template <typename R, int STAGE, bool SLOW>
__device__ __forceinline__ void tm_read(const TmGeom& g, const TmArgs& a, const TmField<R>& f, int kx, int l, int m,
                                        TmVal<R>& v) {
  v.n = tm_N<R, SLOW>(g, f, kx, l, m);
  if constexpr (STAGE == 0) {
    v.x = f.p[f.at(kx, l, m)];
  } else {
    const uint32_t nat = TmField<R>{nullptr, g.nkr, g.ny, g.nz}.at(kx, l, m);
    v.u = reinterpret_cast<const cplx<R>*>(a.sol)[nat];
    v.x = STAGE == 1 ? v.u : f.p[f.at(kx, l, m)];
    v.L = a.L[nat];
    if constexpr (STAGE == 4) {
      const uint32_t pk = f.at(kx, l, m);
      v.r1 = reinterpret_cast<const cplx<R>*>(a.R[0])[pk];
      v.r2 = reinterpret_cast<const cplx<R>*>(a.R[1])[pk];
      v.r3 = reinterpret_cast<const cplx<R>*>(a.R[2])[pk];
      if (a.F) v.F = a.F[nat];
    }
  }
}
template <typename R, int STAGE>
__device__ __forceinline__ void tm_write(const TmGeom& g, const TmArgs& a, int kx, int l, int m, const TmVal<R>& v) {
  const uint32_t nat = TmField<R>{nullptr, g.nkr, g.ny, g.nz}.at(kx, l, m);
  if constexpr (STAGE == 0) {
    reinterpret_cast<cplx<R>*>(a.out)[nat] = v.n;
  } else {
    const cplx<R> r = mkc<R>((R)((double)v.n.x + v.L * (double)v.x.x), (R)((double)v.n.y + v.L * (double)v.x.y));
    if constexpr (STAGE < 4) {
      const uint32_t pk = TmField<R>{nullptr, g.KX, g.KY, g.KZ}.at(kx, l, m);
      reinterpret_cast<cplx<R>*>(a.R[STAGE - 1])[pk] = r;
      reinterpret_cast<cplx<R>*>(a.out)[pk] =
          mkc<R>((R)((double)v.u.x + a.h * (double)r.x), (R)((double)v.u.y + a.h * (double)r.y));
    } else {
      const double sx = (double)v.r1.x + 2.0 * (double)v.r2.x + 2.0 * (double)v.r3.x + (double)r.x;
      const double sy = (double)v.r1.y + 2.0 * (double)v.r2.y + 2.0 * (double)v.r3.y + (double)r.y;
      cplx<R> w = mkc<R>((R)((double)v.u.x + a.h6 * sx), (R)((double)v.u.y + a.h6 * sy));
      if (a.F) w = mkc<R>((R)((double)w.x * v.F), (R)((double)w.y * v.F));
      reinterpret_cast<cplx<R>*>(a.sol)[nat] = w;
    }
  }
}
// 0 where z is finite, else NaN
template <typename R>
__device__ __forceinline__ R tm_nan(cplx<R> z) {
  return z.x * R(0) + z.y * R(0);
}
// one mode; a mode that is not finite is noted, but for the imaginary part of the mean, which c2r ignores
template <typename R, int STAGE, bool SLOW>
__device__ __forceinline__ R tm_mode(const TmGeom& g, const TmArgs& a, const TmField<R>& f, int kx, int l, int m) {
  TmVal<R> v;
  tm_read<R, STAGE, SLOW>(g, a, f, kx, l, m, v);
  tm_write<R, STAGE>(g, a, kx, l, m, v);
  return tm_nan<R>(SLOW && kx == 0 && l == 0 && m == 0 ? mkc<R>(v.x.x, 0) : v.x);
}

// Workgroups: groups of kTmPlanes consecutive m in order, each first the
// columns kx > q in tiles over (l, kx), then the few columns that need the
// kx = 0 plane's symmetry, one mode a thread, so that no wavefront runs both
// forms and none has a long chain of them (four modes a thread there: 140 us
// a step of 256^3 FP32 instead of 109, 41 instead of 21 at 48^3 FP64).  Each XCD
// takes a contiguous range of m: neighbouring planes are read from its L2.
template <typename R, int STAGE>
__global__ void __launch_bounds__(kTmThreads) k_tracer_modes(TmGeom g, TmArgs a) {
  // bad[0] of a run: cleared in its first stage 1, whose finds go to bad[1];
  // stage 2 takes those over and stage 3 clears bad[1], so no launch sets a
  // flag that it clears or reads
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (STAGE == 1 && a.first) a.bad[0] = 0;
    if (STAGE == 2 && a.bad[1]) a.bad[0] = 1;
    if (STAGE == 3) a.bad[1] = 0;
  }
  const int blk = (int)(blockIdx.x % 8) * g.per_xcd + (int)(blockIdx.x / 8);
  if (blk >= g.nblk) return;
  const int tiles = g.tfast + g.tslow;
  const int mg = blk / tiles;
  int tile = blk - mg * tiles;
  const bool slow = tile >= g.tfast;
  if (slow) tile -= g.tfast;
  const int w = slow ? g.slow : g.KX - g.slow;  // columns of this form
  const int idx = tile * kTmThreads + (int)threadIdx.x;
  int row = (int)(((float)idx + 0.5f) * (slow ? g.inv_slow : g.inv_fast));
  const int kx = idx - row * w + (slow ? 0 : g.slow);
  int j = 0;  // plane of the group (a thread of the slow columns takes one)
  if (slow)
    while (row >= g.KY && j < kTmPlanes) {
      row -= g.KY;
      ++j;
    }
  if (row >= g.KY || j >= kTmPlanes) return;
  const int l = row + g.lmin;
  const bool native = STAGE <= 1;
  const TmField<R> f{reinterpret_cast<const cplx<R>*>(a.x), native ? g.nkr : g.KX, native ? g.ny : g.KY,
                     native ? g.nz : g.KZ};
  const int m0 = g.mmin + mg * kTmPlanes, m1 = min(m0 + kTmPlanes - 1, g.mmax);
  R nan = 0;  // stays 0 while every mode is finite
  if (slow) {
    if (m0 + j <= m1) nan = tm_mode<R, STAGE, true>(g, a, f, kx, l, m0 + j);
  } else if (m1 - m0 == kTmPlanes - 1) {
    TmVal<R> v[kTmPlanes];  // all reads before the first store, so that they are in flight together
#pragma unroll
    for (int j = 0; j < kTmPlanes; ++j) tm_read<R, STAGE, false>(g, a, f, kx, l, m0 + j, v[j]);
#pragma unroll
    for (int j = 0; j < kTmPlanes; ++j) {
      tm_write<R, STAGE>(g, a, kx, l, m0 + j, v[j]);
      nan += tm_nan<R>(v[j].x);
    }
  } else {
    for (int m = m0; m <= m1; ++m) nan += tm_mode<R, STAGE, false>(g, a, f, kx, l, m);
  }
  if (nan != R(0)) a.bad[STAGE == 0 ? 2 : STAGE == 1] = 1;
}

__device__ __forceinline__ bool tm_kept(const TmGeom& g, int64_t idx) {
  const int ix = (int)(idx % g.nkr);
  const int64_t r = idx / g.nkr;
  const int iy = (int)(r % g.ny), iz = (int)(r / g.ny);
  return ix < g.KX && (iy <= g.lmax || iy >= g.ny + g.lmin) && (iz <= g.mmax || iz >= g.nz + g.mmin);
}

static __global__ void k_tracer_clear(int* bad) { bad[2] = 0; }

// modes outside the kept band: N = 0; on the band NaN if a mode was not finite
template <typename R>
__global__ void __launch_bounds__(kTmThreads) k_tracer_outside_zero(cplx<R>* N, int64_t total, const int* bad,
                                                                    TmGeom g) {
  const bool fill = bad[2] != 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    if (!tm_kept(g, i))
      N[i] = mkc<R>(0, 0);
    else if (fill)
      N[i] = mkc<R>((R)NAN, (R)NAN);
  }
}

// The same after a run: outside the band the RK4 steps of du/dt = L u, with the
// stages' roundings (zeros stay: all of them where L is finite)
template <typename R>
__global__ void __launch_bounds__(kTmThreads) k_tracer_outside(cplx<R>* sol, const double* L, const double* F,
                                                               double h2, double h, double h6, int64_t nsteps,
                                                               int64_t total, bool zeros_stay, const int* bad,
                                                               TmGeom g) {
  const bool fill = bad[0] != 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    if (tm_kept(g, i)) {
      if (fill) sol[i] = mkc<R>((R)NAN, (R)NAN);
      continue;
    }
    cplx<R> u = sol[i];
    if (zeros_stay && u.x == R(0) && u.y == R(0)) continue;
    const double l = L[i];
    auto rhs = [&](cplx<R> x) { return mkc<R>((R)(l * (double)x.x), (R)(l * (double)x.y)); };
    auto sub = [&](cplx<R> k, double hh) {
      return mkc<R>((R)((double)u.x + hh * (double)k.x), (R)((double)u.y + hh * (double)k.y));
    };
    for (int64_t s = 0; s < nsteps; ++s) {
      const cplx<R> r1 = rhs(u), r2 = rhs(sub(r1, h2)), r3 = rhs(sub(r2, h2)), r4 = rhs(sub(r3, h));
      const double sx = (double)r1.x + 2.0 * (double)r2.x + 2.0 * (double)r3.x + (double)r4.x;
      const double sy = (double)r1.y + 2.0 * (double)r2.y + 2.0 * (double)r3.y + (double)r4.y;
      u = mkc<R>((R)((double)u.x + h6 * sx), (R)((double)u.y + h6 * sy));
      if (F) u = mkc<R>((R)((double)u.x * F[i]), (R)((double)u.y * F[i]));
    }
    sol[i] = u;
  }
}

// ----------------------------------------------------------------- host side
// Boxes of multiples of 2 pi (to rounding: sin and cos are periodic on the
// grid), a dealiased band from which no product aliases back, and layouts that
// 32-bit offsets span; everything else keeps the transforms.
static bool tm_geom(const ffhip_op* op, TmGeom* g) {
  if (op->kind != FFHIP_OP_TRACER3D || op->no_modes || op->spec_count >= (1LL << 30)) return false;
  const double twopi = 6.283185307179586476925286766559;
  int kept[3], kmax[3];
  for (int d = 0; d < 3; ++d) {
    const double r = op->box[d] / twopi, q = std::nearbyint(r);
    if (!(q >= 1) || !(q < 1 << 20) || !(std::fabs(r - q) <= 1e-15 * q)) return false;
    g->q[d] = (int)q;
    const int64_t lo = op->lo[d] - 1, hi = op->hi[d] - 1;  // aliased, 0-based
    if (hi < lo || lo < 1) return false;
    const int64_t neg = d == 0 ? 0 : op->n[d] - 1 - hi;
    if (neg < 0) return false;
    kept[d] = (int)(lo + neg);
    kmax[d] = (int)(lo - 1 > neg ? lo - 1 : neg);
    if (2 * (int64_t)kmax[d] + g->q[d] >= op->n[d]) return false;
    const double x0 = op->params[3 + d];
    if (!std::isfinite(x0) || !std::isfinite(op->params[d])) return false;
    const double amp = 0.5 * op->params[d == 0 ? 1 : d == 1 ? 2 : 0];  // B along x, C along y, A along z
    g->p[d][0] = amp * std::cos(x0);
    g->p[d][1] = amp * std::sin(x0);
  }
  g->nkr = (int)op->nkr;
  g->ny = (int)op->n[1];
  g->nz = (int)op->n[2];
  g->KX = kept[0];
  g->KY = kept[1];
  g->KZ = kept[2];
  g->lmax = (int)op->lo[1] - 2;
  g->lmin = g->lmax + 1 - g->KY;
  g->mmax = (int)op->lo[2] - 2;
  g->mmin = g->mmax + 1 - g->KZ;
  g->slow = g->q[0] + 1 < g->KX ? g->q[0] + 1 : g->KX;
  const int fast = g->KX - g->slow;
  if ((int64_t)g->KX * g->KY * kTmPlanes >= 1 << 20) return false;  // tile indexes divide in FP32
  g->tfast = (fast * g->KY + kTmThreads - 1) / kTmThreads;
  g->tslow = (g->slow * g->KY * kTmPlanes + kTmThreads - 1) / kTmThreads;
  g->inv_fast = fast ? 1.0f / (float)fast : 0.0f;
  g->inv_slow = 1.0f / (float)g->slow;
  g->nblk = (g->tfast + g->tslow) * ((g->KZ + kTmPlanes - 1) / kTmPlanes);
  g->per_xcd = (g->nblk + 7) / 8;
  g->dk = twopi / op->box[0];
  g->dl = twopi / op->box[1];
  g->dm = twopi / op->box[2];
  return true;
}

template <typename R, int STAGE>
static int tm_launch(const TmGeom& g, const TmArgs& a, hipStream_t st) {
  static const char* names[5] = {"tracer_modes", "tracer_modes_stage1", "tracer_modes_stage2", "tracer_modes_stage3",
                                 "tracer_modes_stage4"};
  const double cs = sizeof(cplx<R>), n = (double)g.KX * g.KY * g.KZ;
  const double bytes = n * (STAGE == 0 ? 2 * cs : STAGE == 1 ? 3 * cs + 8 : STAGE < 4 ? 4 * cs + 8 : 6 * cs + 8);
  prof_launch(names[STAGE], bytes, k_tracer_modes<R, STAGE>, dim3(8 * g.per_xcd), dim3(kTmThreads), 0, st, g, a);
  FF_LAUNCHED("k_tracer_modes");
  return FFHIP_OK;
}

template <typename R>
static int tm_calcN(const ffhip_op* op, const TmGeom& g, void* N, const void* sol, hipStream_t st) {
  TmArgs a{};
  a.x = sol;
  a.out = N;
  a.bad = reinterpret_cast<int*>(op->flags);
  hipLaunchKernelGGL(k_tracer_clear, dim3(1), dim3(1), 0, st, a.bad);
  FF_LAUNCHED("k_tracer_clear");
  FF_TRY((tm_launch<R, 0>(g, a, st)));
  hipLaunchKernelGGL((k_tracer_outside_zero<R>), dim3(blocks_for(op->spec_count, kTmThreads, 16384)),
                     dim3(kTmThreads), 0, st, reinterpret_cast<cplx<R>*>(N), op->spec_count, a.bad, g);
  FF_LAUNCHED("k_tracer_outside_zero");
  return FFHIP_OK;
}

// The stage arrays are the operator's transform workspaces, which this path
// leaves free (a packed kept band is smaller than either kind).
template <typename R>
static int tm_rk4(ffhip_op* op, const TmGeom& g, const ffhip_rk4* ts, void* sol, double dt, int64_t nsteps,
                  hipStream_t st) {
  void *s1 = op->spec[0], *s2 = op->spec[1];
  const double h2 = op->prec == FFHIP_F32 ? (double)((float)dt / 2.0f) : dt / 2;
  TmArgs a{};
  a.sol = sol;
  a.R[0] = op->spec[2];
  a.R[1] = op->phys[0];
  a.R[2] = op->phys[1];
  a.L = reinterpret_cast<const double*>(ts->L);
  a.F = reinterpret_cast<const double*>(ts->filter);
  a.h6 = dt / 6;
  a.bad = reinterpret_cast<int*>(op->flags);
  for (int64_t k = 0; k < nsteps; ++k) {
    a.x = sol;
    a.out = s1;
    a.h = h2;
    a.first = k == 0;
    FF_TRY((tm_launch<R, 1>(g, a, st)));
    a.x = s1;
    a.out = s2;
    FF_TRY((tm_launch<R, 2>(g, a, st)));
    a.x = s2;
    a.out = s1;
    a.h = dt;
    FF_TRY((tm_launch<R, 3>(g, a, st)));
    a.x = s1;
    a.out = nullptr;
    FF_TRY((tm_launch<R, 4>(g, a, st)));
  }
  hipLaunchKernelGGL((k_tracer_outside<R>), dim3(blocks_for(op->spec_count, kTmThreads, 16384)), dim3(kTmThreads), 0,
                     st, reinterpret_cast<cplx<R>*>(sol), a.L, a.F, h2, dt, a.h6, nsteps, op->spec_count, ts->L_finite,
                     a.bad, g);
  FF_LAUNCHED("k_tracer_outside");
  return FFHIP_OK;
}

int tracer_modes_calcN(ffhip_op* op, void* N, const void* sol, bool* done, hipStream_t st) {
  TmGeom g;
  *done = tm_geom(op, &g);
  if (!*done) return FFHIP_OK;
  return op->prec == FFHIP_F32 ? tm_calcN<float>(op, g, N, sol, st) : tm_calcN<double>(op, g, N, sol, st);
}

int tracer_modes_rk4(ffhip_op* op, const ffhip_rk4* ts, void* sol, double dt, int64_t nsteps, bool* done,
                     hipStream_t st) {
  TmGeom g;
  *done = !ts->cplx_coef && tm_geom(op, &g);
  if (!*done) return FFHIP_OK;
  return op->prec == FFHIP_F32 ? tm_rk4<float>(op, g, ts, sol, dt, nsteps, st)
                               : tm_rk4<double>(op, g, ts, sol, dt, nsteps, st);
}

}  // namespace ffhip
