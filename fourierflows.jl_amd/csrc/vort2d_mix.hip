// Row and column passes of the fused 2D vorticity steps on the lengths that
// the power-of-two kernels do not take (any other from 16 to 4096 that fits a
// workgroup), with the batched mixed-radix transforms of mix_fft.h.  Layouts, stage
// arithmetic and launch order are those of vort2d_fused.hip; one axis may run
// here and the other there.
//
//   column pass: C adjacent kx columns per workgroup.  Both forward
//     transforms run as one tile of 2 C, the stage combination leaves the new
//     state in LDS, and the three inverse transforms read it as one tile of
//     3 C whose first pass forms zeta^, u^ and v^: two transforms in the
//     serial chain instead of five.  Where 4 C columns do not fit LDS the
//     fields take turns in a tile of C.
//   row pass: a pair of rows per tile (u + iv of each, zeta of both packed in
//     one), three inverse and two forward transforms; a row alone (u + iv and
//     zeta) where three do not fit.
//
// RK4 step on MI355X, plan-based path -> here: 768 x 480 FP64 543 -> 119 us
// (FP32 675 -> 98), 96^2 FP64 418 -> 70 us, 1000 x 750 FP64 665 -> 202 us,
// 1806 x 64 FP32 (a prime factor 43) 6640 -> 160 us.  A launch is bound by the
// latency of its six to eight passes: at 768 x 480 FP64 the columns issue 1.8 us
// of VALU instructions in 15.5 and the rows 3.2 in 14.0, with 1 and 1.4
// wavefronts per SIMD that wait two to three times as long as they issue.
#include "mix_fft.h"
#include "vort2d_body.h"

namespace ffhip {

template <typename R>
__device__ __forceinline__ cplx<R> vstage_any(const int stage, const VortColArgs& a, const int64_t si,
                                              const cplx<R> n) {
  switch (stage) {  // uniform over the launch
    case 0: return vstage_point<R, 0>(a, si, n);
    case 1: return vstage_point<R, 1>(a, si, n);
    case 2: return vstage_point<R, 2>(a, si, n);
    case 3: return vstage_point<R, 3>(a, si, n);
    case 4: return vstage_point<R, 4>(a, si, n);
    default: return vstage_point<R, kVExplicit>(a, si, n);
  }
}

// columns of the blocked arrays, which lie one after the other fd elements
// apart: transform q is column q mod C of array q / C
template <typename R, typename P>
struct VColMem {
  static constexpr bool linear = true;
  P p;
  int lc;
  uint32_t ibase, fd;
  __device__ __forceinline__ bool ok(int, int) const { return true; }
  __device__ __forceinline__ uint32_t base(int, int q, int i) const {
    const uint32_t fl = (uint32_t)q >> lc;
    return (ibase + fl * fd + (uint32_t)i * kVCB + ((uint32_t)q - (fl << lc))) * (uint32_t)sizeof(cplx<R>);
  }
  __device__ __forceinline__ uint32_t step(int d) const { return (uint32_t)(d * kVCB) * (uint32_t)sizeof(cplx<R>); }
  __device__ __forceinline__ cplx<R> get(uint32_t o) const {
    return *reinterpret_cast<const cplx<R>*>(reinterpret_cast<const char*>(p) + o);
  }
  __device__ __forceinline__ void put(uint32_t o, cplx<R> v) const {
    *reinterpret_cast<cplx<R>*>(reinterpret_cast<char*>(p) + o) = v;
  }
};

// C = 1 << lc columns; together: all fields of a direction in one tile
template <typename R, bool PRIME>
__global__ void __launch_bounds__(kMixThreads) k_mvcol(VortGeom g, VortColArgs a, MixDev f, int stage, int lc,
                                                      int together) {
  extern __shared__ unsigned char vsm[];
  __shared__ int table[kMixTable / 4];
  mix_table(f, table, threadIdx.x);
  constexpr int CB = kVCB;
  const int C = 1 << lc;
  int tx, sub;
  xcd_split(blockIdx.x, CB >> lc, &tx, &sub);
  if (tx >= g.TX) return;  // grid is rounded up to whole XCD groups
  const int ny = f.n, tid = threadIdx.x, nt = blockDim.x;
  cplx<R>* tile = reinterpret_cast<cplx<R>*>(vsm);
  cplx<R>* wb = tile + (together ? 3 : 1) * C * ny;  // new state, [ny][C]
  cplx<R>* qb = wb + C * ny;                         // (l, kx) / |k|^2 there
  const uint32_t ibase = (uint32_t)tx * ny * CB + (sub << lc);
  const int ix0 = tx * CB + (sub << lc);
  const uint32_t fd = (uint32_t)g.TX * ny * CB;  // O1 follows O0, and I1, I2 follow I0 (vstate_alloc)
  // forward transforms, (i, c) at i * AS + c: side by side in one tile, or
  // one in wb and one in the tile
  const cplx<R>* A = together ? tile : wb;
  const cplx<R>* B = together ? tile + C : tile;
  const int AS = together ? 2 * C : C;
  if (stage > 0) {
#pragma unroll 1
    for (int b = together; b < 2; ++b) {
      const MixTile<R> T{together || b == 1 ? tile : wb, AS, ny};
      mix_fft<-1, false, R, PRIME>(f, table, T, 1, tid, nt,
                                   VColMem<R, const void*>{a.O0, lc, together ? ibase : ibase + b * fd, fd}, T);
    }
  }
#pragma unroll 1
  for (int idx = tid; idx < C * ny; idx += nt) {
    const int c = idx & (C - 1), iy = idx >> lc;
    const int ix = ix0 + c;
    cplx<R> w = mkc<R>(0, 0), q = mkc<R>(0, 0);
    if (ix < g.KX && (iy < g.ylo || iy > g.yhi)) {
      const R kx = (R)(g.dk * (double)ix), l = (R)(g.dl * (double)vfreq(iy, ny));
      cplx<R> n = mkc<R>(0, 0);
      if (stage > 0) {
        const cplx<R> pa = A[iy * AS + c], pb = B[iy * AS + c];
        n = mkc<R>(kx * pa.y + l * pb.y, -(kx * pa.x) - l * pb.x);  // -i kr A - i l B
      }
      w = vstage_any<R>(stage, a, (int64_t)tx * g.KY * CB + (sub << lc) + c + (int64_t)v_ky(iy, g) * CB, n);
      const R invK = ix == 0 && iy == 0 ? R(0) : R(1) / (kx * kx + l * l);
      q = mkc<R>(l * invK, kx * invK);
    }
    wb[idx] = w;  // this thread's own A where the fields take turns
    qb[idx] = q;
  }
  if (!a.do_inverse) return;  // uniform over the block
  __syncthreads();
  auto field = [&](int fl, int c, int i) {  // zeta^, u^ = i l/|k|^2 zeta^, v^ = -i kr/|k|^2 zeta^
    const cplx<R> z = wb[(i << lc) + c];
    if (fl == 0) return z;
    const cplx<R> q = qb[(i << lc) + c];
    return fl == 1 ? mkc<R>(-q.x * z.y, q.x * z.x) : mkc<R>(q.y * z.y, -q.y * z.x);
  };
#pragma unroll 1
  for (int b = together ? 2 : 0; b < 3; ++b) {  // all three at once, or one after the other
    const int f0 = together ? 0 : b;
    mix_fft<1, false, R, PRIME>(f, table, MixTile<R>{tile, together ? 3 * C : C, ny}, 1, tid, nt,
                                mix_fn([&](int, int q, int i) { return field(f0 + (q >> lc), q & (C - 1), i); }),
                                VColMem<R, void*>{a.I0, lc, ibase + f0 * fd, fd});
    __syncthreads();  // the tile's last reads before it is filled again
  }
}

// ng tiles of a row pair (pair) or of one row per workgroup
template <typename R, bool PRIME>
__global__ void __launch_bounds__(kMixThreads) k_mvrow(VortGeom g, VortRowArgs a, MixDev f, int pair, int ng) {
  extern __shared__ unsigned char vsm[];
  __shared__ int table[kMixTable / 4];
  mix_table(f, table, threadIdx.x);
  constexpr int CB = kVCB;
  const int nx = f.n, tid = threadIdx.x, nt = blockDim.x;
  const int RG = pair ? 2 : 1;  // rows per tile
  const int y0 = blockIdx.x * RG * ng;
  const uint32_t ny = (uint32_t)g.ny;
  const int KX = g.KX;
  cplx<R>* lds = reinterpret_cast<cplx<R>*>(vsm);
  auto iaddr = [&](int k, int y) -> uint32_t {
    return ((uint32_t)(k / CB) * ny + (uint32_t)y) * CB + (uint32_t)(k % CB);
  };
  const cplx<R>* Zh = reinterpret_cast<const cplx<R>*>(a.I0);
  const cplx<R>* Uh = reinterpret_cast<const cplx<R>*>(a.I1);
  const cplx<R>* Vh = reinterpret_cast<const cplx<R>*>(a.I2);
  const MixTile<R> T3{lds, RG + 1, nx};
  // A + i B of two Hermitian-extended half spectra: (u^, v^) of a row, or
  // zeta^ of the tile's rows; c2r ignores Im at kx = 0
  mix_fft<1, false, R, PRIME>(
      f, table, T3, ng, tid, nt,
      mix_fn([&](int tg, int q, int i) {
        const int y = y0 + tg * RG;
        if (y >= (int)ny) return mkc<R>(0, 0);
        const bool lo = i < KX, hi = i > nx - KX;
        if (!lo && !hi) return mkc<R>(0, 0);
        const int kk = lo ? i : nx - i;
        const bool zt = q == RG;
        const cplx<R> p = at32(zt ? Zh : Uh, iaddr(kk, zt ? y : y + q));
        cplx<R> s = mkc<R>(0, 0);
        if (!zt || pair) s = at32(zt ? Zh : Vh, iaddr(kk, zt ? y + 1 : y + q));
        const R py = i == 0 ? R(0) : (lo ? p.y : -p.y), sy = i == 0 ? R(0) : (lo ? s.y : -s.y);
        return mkc<R>(p.x - sy, py + s.x);
      }),
      T3);
  // products and the forward transform of u zeta + i v zeta
  const MixTile<R> T2{lds, RG, nx};
  const R s2 = (R)g.s2;
  mix_fft<-1, true, R, PRIME>(
      f, table, T2, ng, tid, nt,
      mix_fn([&](int tg, int q, int i) {
        const cplx<R> uv = T3.at(tg, q, i), z = T3.at(tg, RG, i);
        const R zz = (q == 0 ? z.x : z.y) * s2;
        return mkc<R>(uv.x * zz, uv.y * zz);
      }),
      T2);
  // split W into the half spectra of its real and imaginary parts
  cplx<R>* O0 = reinterpret_cast<cplx<R>*>(a.O0);
  cplx<R>* O1 = reinterpret_cast<cplx<R>*>(a.O1);
  const int rows = RG * ng;
  const float inv_rows = 1.0f / (float)rows;
  for (int idx = tid; idx < g.KXp * rows; idx += nt) {
    const int rest = idx / CB;
    const int kb = mix_div(rest, inv_rows);
    const int r = rest - kb * rows, k = kb * CB + idx % CB;
    if (y0 + r >= (int)ny) continue;
    const int tg = pair ? r >> 1 : r, q = pair ? r & 1 : 0;
    cplx<R> Pk = mkc<R>(0, 0), Qk = mkc<R>(0, 0);
    if (k < KX) {
      const cplx<R> wk = T2.at(tg, q, k);
      const cplx<R> wc = cconj<R>(T2.at(tg, q, k == 0 ? 0 : nx - k));
      Pk = mkc<R>(R(0.5) * (wk.x + wc.x), R(0.5) * (wk.y + wc.y));
      Qk = mkc<R>(R(0.5) * (wk.y - wc.y), -R(0.5) * (wk.x - wc.x));  // (wk - wc) / (2i)
    }
    const uint32_t o = iaddr(k, y0 + r);
    at32(O0, o) = Pk;
    at32(O1, o) = Qk;
  }
}

// ----------------------------------------------------------------- host side
static size_t vcol_bytes(int prec, int n, int C, bool together) {
  return (size_t)(together ? 5 : 3) * C * n * cplx_size(prec);
}

bool mix_vcol_ok(int prec, int64_t n, MixFft* f) {
  return mix_schedule(n, f) && mix_threads(*f, 1) > 0 && vcol_bytes(prec, (int)n, 1, false) <= kMixLds;
}
bool mix_vrow_ok(int prec, int64_t n, MixFft* f) {
  return mix_schedule(n, f) && mix_threads(*f, 2) > 0 && mix_lds(*f, 2, prec) <= kMixLds;
}

// twice the threads while that leaves the launch within two wavefronts per
// SIMD (what the FP64 kernels' registers allow at once: 1000 x 750 FP64 201 us
// a step so, 235 us with three) and a pass has butterflies for them
static int more_threads(const MixFft& f, int B, int t, int64_t wgs) {
  int most = 0;
  for (int i = 0; i < f.npass; ++i) most = f.p[i].m > most ? f.p[i].m : most;
  while (2 * t <= kMixThreads && 2 * t <= (B * most + 63) / 64 * 64 && wgs * 2 * t / 64 <= 2048) t *= 2;
  return t;
}

template <typename R>
static int mvcol(const VortGeom& g, const MixFft& f, const void* tw, int stage, const VortColArgs& a, hipStream_t st) {
  constexpr int prec = sizeof(R) == 4 ? FFHIP_F32 : FFHIP_F64;
  auto kern = mix_prime_pass(f) ? k_mvcol<R, true> : k_mvcol<R, false>;
  static bool attr[2] = {false, false};
  FF_TRY(mix_lds_attr(kern, &attr[mix_prime_pass(f)]));
  auto fits = [&](int C, bool tog) {
    return vcol_bytes(prec, f.n, C, tog) <= kMixLds && mix_threads(f, (tog ? 3 : 1) * C) > 0;
  };
  int lc = 0;
  const bool tog = fits(1, true);
  // two and four columns per workgroup while that leaves one for every compute
  // unit (768 x 480 FP32: 98 us a step, 111 us with four columns on 64 units)
  while (lc < 2 && fits(2 << lc, tog) && vcol_bytes(prec, f.n, 2 << lc, tog) <= kMixLds / 2 &&
         g.TX * (kVCB >> (lc + 1)) >= 256)
    ++lc;
  const int B = (tog ? 3 : 1) << lc;
  const int groups = (g.TX + kXCD - 1) / kXCD * kXCD;
  const int nb = groups * (kVCB >> lc);
  static const char* names[6] = {"vort_col_stage0", "vort_col_stage1", "vort_col_stage2", "vort_col_stage3",
                                 "vort_col_stage4", "vort_col_explicit"};
  prof_launch(names[stage], col_bytes<R>(g, stage, a.do_inverse), kern, dim3(nb),
              dim3(more_threads(f, B, mix_threads(f, B), nb)), vcol_bytes(prec, f.n, 1 << lc, tog), st, g, a, mix_dev(f, tw), stage, lc, tog ? 1 : 0);
  FF_LAUNCHED("k_mvcol");
  return FFHIP_OK;
}

template <typename R>
static int mvrow(const VortGeom& g, const MixFft& f, const void* tw, const VortRowArgs& a, hipStream_t st) {
  constexpr int prec = sizeof(R) == 4 ? FFHIP_F32 : FFHIP_F64;
  auto kern = mix_prime_pass(f) ? k_mvrow<R, true> : k_mvrow<R, false>;
  static bool attr[2] = {false, false};
  FF_TRY(mix_lds_attr(kern, &attr[mix_prime_pass(f)]));
  const int pair = mix_threads(f, 3) > 0 && mix_lds(f, 3, prec) <= kMixLds;
  const int G = pair ? 3 : 2;
  int ng = 1;
  while (mix_threads(f, G * (ng + 1)) > 0 && mix_lds(f, G * (ng + 1), prec) <= kMixLds / 2 &&
         G * (ng + 1) * f.n <= 3072 && g.ny >= (G - 1) * (ng + 1) * 512)
    ++ng;
  const int rows = (G - 1) * ng;
  const int nb = (g.ny + rows - 1) / rows;
  prof_launch("vort_row", row_bytes<R>(g), kern, dim3(nb),
              dim3(more_threads(f, G * ng, mix_threads(f, G * ng), nb)), mix_lds(f, G * ng, prec), st, g, a, mix_dev(f, tw), pair, ng);
  FF_LAUNCHED("k_mvrow");
  return FFHIP_OK;
}

int mix_vcol(int prec, const VortGeom& g, const MixFft& f, const void* tw, int stage, const VortColArgs& a,
             hipStream_t st) {
  return prec == FFHIP_F32 ? mvcol<float>(g, f, tw, stage, a, st) : mvcol<double>(g, f, tw, stage, a, st);
}
int mix_vrow(int prec, const VortGeom& g, const MixFft& f, const void* tw, const VortRowArgs& a, hipStream_t st) {
  return prec == FFHIP_F32 ? mvrow<float>(g, f, tw, a, st) : mvrow<double>(g, f, tw, a, st);
}

}  // namespace ffhip
