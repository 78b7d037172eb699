// Mixed-radix kernels of the FFT plans (mul!/ldiv!, src/domains.jl:2-5): the
// axes that the power-of-two kernels of fft_fast.hip do not take (any other
// length, rows of the complex plans, and the powers of two below and above
// their range), as long as a transform fits one LDS tile and one workgroup.
//
// Against the Stockham kernels of fft.hip (two tiles in LDS, radices up to 8
// or a direct prime, run-time divisions), mul! plus ldiv! on MI355X: 1000 x
// 750 FP64 58 -> 32 us, 192^3 FP32 190 -> 110 us and FP64 274 -> 155 us,
// 1536^2 FP32 80 -> 45 us, 360^2 FP32 47 -> 24 us, 512 x 4096 FP64 124 -> 66
// us, complex 1024^2 FP32 43 -> 33 us.  The grids of a few megabytes are bound
// by the latency of their passes (1000 x 750 FP64: 1.5 us of VALU issue at most
// in 7 to 10, about one wavefront per SIMD).  At 192^3 the columns are bound by
// memory (4.3 to 4.5 TB/s; a line that two workgroups share is fetched twice),
// the rows by LDS, where bank conflicts take 66 to 79% of its cycles.
#include <cstdlib>
#include <cstring>
#include <utility>

#include "mix_fft.h"
#include "plan.h"
#include "prof.h"

namespace ffhip {

// ----------------------------------------------------------------- schedules
static const int kRadices[] = {16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

static void mix_search(int64_t n, int depth, int maxrad, int* cur, int* best, int* nbest, int* cost) {
  if (n == 1) {
    int sum = 0;
    bool odd = false;
    for (int i = 0; i < depth; ++i) {
      sum += cur[i];
      odd |= cur[i] % 2 == 1;
    }
    sum += depth * 1000 + (odd ? 0 : 8);  // fewest passes, then an odd radix for the first, then the smallest radices
    if (*nbest == 0 || sum < *cost) {
      *cost = sum;
      *nbest = depth;
      for (int i = 0; i < depth; ++i) best[i] = cur[i];
    }
    return;
  }
  if (depth == kMixMaxPass) return;
  for (int r : kRadices) {
    if (r > maxrad || n % r) continue;
    cur[depth] = r;
    mix_search(n / r, depth + 1, r, cur, best, nbest, cost);
  }
}

bool mix_schedule(int64_t n, MixFft* f) {
  if (n < 2 || n > (1 << 15)) return false;
  int rad[kMixMaxPass + 8], big[8], np = 0, nbig = 0;
  int64_t m = n;
  for (int p : {2, 3, 5, 7, 11, 13})
    while (m % p == 0) m /= p;
  int64_t smooth = n / m;
  for (int64_t p = 17; m > 1; p += 2)  // at most three factors of 17 and more
    while (m % p == 0 || (m > 1 && p * p > m)) {
      const int64_t q = m % p == 0 ? p : m;
      if (q > kMixPrime) return false;
      big[nbig++] = (int)q;
      m /= q;
    }
  if (smooth > 1) {
    int cur[kMixMaxPass], cost = 0;
    mix_search(smooth, 0, 16, cur, rad, &np, &cost);
    if (np == 0) return false;
  } else {
    rad[np++] = 1;  // primes act on the tile: a copying pass brings the points there
  }
  if (np == 1 && nbig == 0) {  // a pass of its own reads and one writes the tile: two passes at least
    for (int a = 2; a * a <= smooth && np == 1; ++a)
      if (smooth % a == 0) {
        rad[0] = (int)smooth / a;
        rad[1] = a;
        np = 2;
      }
    if (np == 1) return false;
  }
  // an odd radix first, else one that is twice an odd number, else the smallest
  auto rank = [](int r) { return r % 2 ? 0 : r % 4 ? 1 : 2; };
  for (int i = 1; i < np; ++i)
    if (rank(rad[i]) < rank(rad[0]) || (rank(rad[i]) == 2 && rank(rad[0]) == 2 && rad[i] < rad[0]))
      std::swap(rad[0], rad[i]);
  for (int i = 0; i < nbig; ++i) rad[np++] = big[i];
  if (np > kMixMaxPass) return false;
  f->n = (int)n;
  f->npass = np;
  int Ns = 1, tw = 0;
  for (int i = 0; i < np; ++i) {
    MixPass& p = f->p[i];
    p.rad = rad[i];
    p.Ns = Ns;
    p.m = (int)n / rad[i];
    p.tw = tw;
    p.inv_m = 1.0f / (float)p.m;
    p.inv_Ns = 1.0f / (float)Ns;
    if (Ns > 1) tw += (rad[i] - 1) * Ns;
    if (rad[i] > 16) tw += rad[i];  // its own roots of unity
    Ns *= rad[i];
  }
  return true;
}

int mix_upload(const MixFft& f, int prec, void** dptr) {
  std::vector<double> h;
  auto root = [&](int64_t k, int64_t n) {
    double c, s;
    unit_root(k, n, &c, &s);
    h.push_back(c);
    h.push_back(-s);
  };
  for (int i = 0; i < f.npass; ++i) {
    const MixPass& p = f.p[i];
    if (p.Ns > 1)
      for (int r = 1; r < p.rad; ++r)
        for (int k = 0; k < p.Ns; ++k) root((int64_t)r * k, (int64_t)p.Ns * p.rad);
    if (p.rad > 16)
      for (int e = 0; e < p.rad; ++e) root(e, p.rad);
  }
  std::vector<char> buf(kMixTable + h.size() / 2 * cplx_size(prec), 0);
  std::memcpy(buf.data(), f.p, f.npass * sizeof(MixPass));
  if (prec == FFHIP_F64) {
    std::memcpy(buf.data() + kMixTable, h.data(), h.size() * sizeof(double));
  } else {
    float* s = reinterpret_cast<float*>(buf.data() + kMixTable);
    for (size_t i = 0; i < h.size(); ++i) s[i] = (float)h[i];
  }
  FF_TRY(dev_alloc(dptr, buf.size()));
  FF_HIP(hipMemcpy(*dptr, buf.data(), buf.size(), hipMemcpyHostToDevice));
  return FFHIP_OK;
}

int mix_threads(const MixFft& f, int64_t B) {
  int64_t t = 1;
  for (int i = 0; i < f.npass; ++i) {
    const int rad = f.p[i].rad;  // a prime's threads take two units of four output pairs
    const int64_t bf = rad > 16 ? B * f.p[i].m * ((rad - 1) / 8 + 1) : B * f.p[i].m, nb = rad > 16 ? 2 : mix_nbf(rad);
    if ((bf + nb - 1) / nb > t) t = (bf + nb - 1) / nb;
  }
  t = (t + 63) / 64 * 64;
  return t <= kMixThreads && B * f.n < (1 << 20) ? (int)t : 0;
}

// ----------------------------------------------------------------- kernels
// Tile geometry of one launch: B = ng * G transforms per workgroup
struct MixShape {
  int G, ng;
};

// c2c of contiguous rows
template <int DIR, typename R, bool PRIME>
__global__ void __launch_bounds__(kMixThreads) k_mrows_c2c(const cplx<R>* __restrict__ in, cplx<R>* __restrict__ out,
                                                          MixDev f, int64_t nrows, MixShape sh, R scale) {
  extern __shared__ unsigned char msm[];
  __shared__ int table[kMixTable / 4];
  mix_table(f, table, threadIdx.x);
  const MixTile<R> T{reinterpret_cast<cplx<R>*>(msm), sh.G, f.n};
  const int64_t row0 = (int64_t)blockIdx.x * sh.G * sh.ng;
  const int left = (int)(nrows - row0 < sh.G * sh.ng ? nrows - row0 : sh.G * sh.ng);
  const uint32_t n = (uint32_t)f.n;
  mix_fft<DIR, false, R, PRIME>(f, table, T, sh.ng, threadIdx.x, blockDim.x,
                         MixMem<R, const cplx<R>*>{in + row0 * n, sh.G, left, n, 1, R(1)},
                         MixMem<R, cplx<R>*>{out + row0 * n, sh.G, left, n, 1, scale});
}

// r2c of contiguous rows of 2m reals read as m complex pairs, split into m + 1 coefficients
template <typename R, bool PRIME>
__global__ void __launch_bounds__(kMixThreads) k_mrows_r2c(const cplx<R>* __restrict__ in, cplx<R>* __restrict__ out,
                                                          MixDev f, const cplx<R>* __restrict__ rtw, int64_t nrows,
                                                          MixShape sh) {
  extern __shared__ unsigned char msm[];
  __shared__ int table[kMixTable / 4];
  mix_table(f, table, threadIdx.x);
  const MixTile<R> T{reinterpret_cast<cplx<R>*>(msm), sh.G, f.n};
  const int m = f.n;
  const int64_t row0 = (int64_t)blockIdx.x * sh.G * sh.ng;
  const int left = (int)(nrows - row0 < sh.G * sh.ng ? nrows - row0 : sh.G * sh.ng);
  mix_fft<-1, false, R, PRIME>(f, table, T, sh.ng, threadIdx.x, blockDim.x,
                        MixMem<R, const cplx<R>*>{in + row0 * m, sh.G, left, (uint32_t)m, 1, R(1)}, T);
  const int nk = m + 1;
  const float inv_nk = 1.0f / (float)nk, inv_G = 1.0f / (float)sh.G;
  cplx<R>* dst = out + row0 * nk;
  for (int i = threadIdx.x; i < left * nk; i += blockDim.x) {
    const int t = mix_div(i, inv_nk);
    const int k = i - t * nk;
    const int tg = mix_div(t, inv_G), g = t - tg * sh.G;
    const cplx<R> zk = T.at(tg, g, k == m ? 0 : k);
    const cplx<R> zc = cconj<R>(T.at(tg, g, k == 0 ? 0 : m - k));
    const cplx<R> xe = cscale<R>(cadd<R>(zk, zc), R(0.5));
    const cplx<R> d = csub<R>(zk, zc);
    const cplx<R> xo = mkc<R>(R(0.5) * d.y, -R(0.5) * d.x);  // (zk - zc) / (2i)
    at32(dst, (uint32_t)i) = cadd<R>(xe, cmul<R>(at32(rtw, (uint32_t)k), xo));
  }
}

// c2r of contiguous rows: m + 1 coefficients to 2m reals, scaled
template <typename R, bool PRIME>
__global__ void __launch_bounds__(kMixThreads) k_mrows_c2r(const cplx<R>* __restrict__ in, cplx<R>* __restrict__ out,
                                                          MixDev f, const cplx<R>* __restrict__ rtw, int64_t nrows,
                                                          MixShape sh, R scale) {
  extern __shared__ unsigned char msm[];
  __shared__ int table[kMixTable / 4];
  mix_table(f, table, threadIdx.x);
  const MixTile<R> T{reinterpret_cast<cplx<R>*>(msm), sh.G, f.n};
  const int m = f.n;
  const int64_t row0 = (int64_t)blockIdx.x * sh.G * sh.ng;
  const int left = (int)(nrows - row0 < sh.G * sh.ng ? nrows - row0 : sh.G * sh.ng);
  const cplx<R>* src = in + row0 * (m + 1);
  mix_fft<1, false, R, PRIME>(f, table, T, sh.ng, threadIdx.x, blockDim.x, mix_fn([&](int tg, int g, int k) {
                         const int t = min(tg * sh.G + g, left - 1);
                         cplx<R> xk = at32(src, (uint32_t)(t * (m + 1) + k));
                         cplx<R> xm = at32(src, (uint32_t)(t * (m + 1) + m - k));
                         if (k == 0) {  // imaginary parts of DC and Nyquist are ignored
                           xk.y = 0;
                           xm.y = 0;
                         }
                         const cplx<R> xmc = cconj<R>(xm);
                         const cplx<R> xe = cscale<R>(cadd<R>(xk, xmc), R(0.5));
                         const cplx<R> xo =
                             cmul<R>(cscale<R>(csub<R>(xk, xmc), R(0.5)), cconj<R>(at32(rtw, (uint32_t)k)));
                         return mkc<R>(xe.x - xo.y, xe.y + xo.x);  // xe + i xo
                       }),
                       MixMem<R, cplx<R>*>{out + row0 * m, sh.G, left, (uint32_t)m, 1, scale});
}

// c2c along a strided axis: transform (slab, column c) has element i at
// slab * slab_dist + c + i * stride; a workgroup takes G * ng adjacent columns
// (in and out may be the same array: a workgroup reads its columns before it
// writes them).  Each XCD takes a contiguous range of per_xcd workgroups, so
// that the lines two of them share stay in one L2; per_xcd = 0: in order.
template <int DIR, typename R, bool PRIME>
__global__ void __launch_bounds__(kMixThreads) k_mcols(const cplx<R>* in, cplx<R>* out, MixDev f, int64_t ncols,
                                                      uint32_t stride, int64_t slab_dist, MixShape sh, R scale,
                                                      int per_xcd) {
  extern __shared__ unsigned char msm[];
  __shared__ int table[kMixTable / 4];
  mix_table(f, table, threadIdx.x);
  const MixTile<R> T{reinterpret_cast<cplx<R>*>(msm), sh.G, f.n};
  const int64_t blk = per_xcd ? (int64_t)(blockIdx.x % 8) * per_xcd + blockIdx.x / 8 : blockIdx.x;
  const int64_t col0 = blk * sh.G * sh.ng;
  if (col0 >= ncols) return;  // whole workgroup, before any barrier
  const int left = (int)(ncols - col0 < sh.G * sh.ng ? ncols - col0 : sh.G * sh.ng);
  const int64_t base = (int64_t)blockIdx.y * slab_dist + col0;
  mix_fft<DIR, false, R, PRIME>(f, table, T, sh.ng, threadIdx.x, blockDim.x,
                         MixMem<R, const cplx<R>*>{in + base, sh.G, left, 1, stride, R(1)},
                         MixMem<R, cplx<R>*>{out + base, sh.G, left, 1, stride, scale});
}

// ----------------------------------------------------------------- host side
// one transform fits a workgroup
bool mix_fits(const MixFft& f, int prec) { return mix_threads(f, 1) > 0 && mix_lds(f, 1, prec) <= kMixLds; }

// Transforms per workgroup.  Columns start at gmin adjacent ones (32 B of a
// row) and take more, up to whole 128 B lines, only while that leaves 512
// workgroups, two for each compute unit: fewer leave the chip idle (768 x 480
// FP64 mul! + ldiv!: 35 us with the groups filled first, 30 us so).  Short
// rows and columns fill a tile of 1024 elements (192^3 FP32: 1024 and 2048
// measure the same, 4096 is 4% slower); rows up to 256 elements do so on any
// number of workgroups, since a wavefront of its own for 8 points is mostly
// launch (mul! of 16 x 2048 FP32, half length 8: 11.9 us -> 11.5 us).
static MixShape shape(const MixFft& f, int prec, int64_t count, int64_t total, int gmin, int gmax) {
  constexpr int64_t kElems = 1024, kWgs = 512, kRow = 256;
  MixShape s{1, 1};
  while (s.G * 2 <= gmax && s.G < count && mix_threads(f, 2 * s.G) > 0 && mix_lds(f, 2 * s.G, prec) <= kMixLds / 2 &&
         (s.G < gmin || total >= 2 * s.G * kWgs))
    s.G *= 2;
  while ((int64_t)s.G * s.ng < count && (int64_t)s.G * (s.ng + 1) * f.n <= kElems &&
         (total >= (int64_t)s.G * (s.ng + 1) * kWgs || (gmax == 1 && (int64_t)(s.ng + 1) * f.n <= kRow)) &&
         mix_threads(f, s.G * (s.ng + 1)) > 0)
    ++s.ng;
  return s;
}

// Threads: enough to hold the tile, and twice that (again and again) while
// the launch has under two wavefronts per SIMD and a pass has butterflies for
// them: fewer points per thread shorten each pass (1000 x 750 FP64: 38.8 ->
// 36.4 us).
int mix_wg_threads(const MixFft& f, int B, int64_t wgs) {
  int w = mix_threads(f, B), most = 0;
  for (int i = 0; i < f.npass; ++i) most = f.p[i].m > most ? f.p[i].m : most;
  while (2 * w <= kMixThreads && 2 * w <= (B * most + 63) / 64 * 64 && wgs * w / 64 < 2048) w *= 2;
  return w;
}

static MixShape row_shape(const MixFft& f, int prec, int64_t nrows) {
  return shape(f, prec, nrows, nrows, 1, 1);
}

template <typename R, int DIR>
static int rows_c2c_t(const void* in, void* out, int64_t nrows, const Axis& ax, double scale, hipStream_t st) {
  const int prec = prec_code<R>();
  const MixShape s = row_shape(ax.mix, prec, nrows);
  const int B = s.G * s.ng;
  auto kern = mix_prime_pass(ax.mix) ? k_mrows_c2c<DIR, R, true> : k_mrows_c2c<DIR, R, false>;
  static bool attr[2] = {false, false};
  FF_TRY(mix_lds_attr(kern, &attr[mix_prime_pass(ax.mix)]));
  prof_launch("fft_rows_c2c", 2.0 * nrows * ax.n * sizeof(cplx<R>), kern,
              dim3((unsigned)((nrows + B - 1) / B)), dim3(mix_wg_threads(ax.mix, B, (nrows + B - 1) / B)), mix_lds(ax.mix, B, prec), st,
              reinterpret_cast<const cplx<R>*>(in), reinterpret_cast<cplx<R>*>(out), mix_dev(ax.mix, ax.mixtw), nrows, s, (R)scale);
  FF_LAUNCHED("k_mrows_c2c");
  return FFHIP_OK;
}

template <typename R>
static int rows_r2c_t(const void* in, void* out, int64_t nrows, const Axis& ax, const void* rtw, hipStream_t st) {
  const int prec = prec_code<R>();
  const MixShape s = row_shape(ax.mix, prec, nrows);
  const int B = s.G * s.ng;
  auto kern = mix_prime_pass(ax.mix) ? k_mrows_r2c<R, true> : k_mrows_r2c<R, false>;
  static bool attr[2] = {false, false};
  FF_TRY(mix_lds_attr(kern, &attr[mix_prime_pass(ax.mix)]));
  prof_launch("fft_rows_r2c", (double)nrows * (2.0 * ax.n + 1) * sizeof(cplx<R>), kern,
              dim3((unsigned)((nrows + B - 1) / B)), dim3(mix_wg_threads(ax.mix, B, (nrows + B - 1) / B)), mix_lds(ax.mix, B, prec), st,
              reinterpret_cast<const cplx<R>*>(in), reinterpret_cast<cplx<R>*>(out), mix_dev(ax.mix, ax.mixtw), reinterpret_cast<const cplx<R>*>(rtw), nrows, s);
  FF_LAUNCHED("k_mrows_r2c");
  return FFHIP_OK;
}

template <typename R>
static int rows_c2r_t(const void* in, void* out, int64_t nrows, const Axis& ax, const void* rtw, double scale,
                      hipStream_t st) {
  const int prec = prec_code<R>();
  const MixShape s = row_shape(ax.mix, prec, nrows);
  const int B = s.G * s.ng;
  auto kern = mix_prime_pass(ax.mix) ? k_mrows_c2r<R, true> : k_mrows_c2r<R, false>;
  static bool attr[2] = {false, false};
  FF_TRY(mix_lds_attr(kern, &attr[mix_prime_pass(ax.mix)]));
  prof_launch("fft_rows_c2r", (double)nrows * (2.0 * ax.n + 1) * sizeof(cplx<R>), kern,
              dim3((unsigned)((nrows + B - 1) / B)), dim3(mix_wg_threads(ax.mix, B, (nrows + B - 1) / B)), mix_lds(ax.mix, B, prec), st,
              reinterpret_cast<const cplx<R>*>(in), reinterpret_cast<cplx<R>*>(out), mix_dev(ax.mix, ax.mixtw), reinterpret_cast<const cplx<R>*>(rtw), nrows, s, (R)scale);
  FF_LAUNCHED("k_mrows_c2r");
  return FFHIP_OK;
}

template <typename R, int DIR>
static int cols_t(const void* in, void* out, int64_t ncols, int64_t stride, int64_t nslabs, int64_t slab_dist,
                  const Axis& ax, double scale, hipStream_t st) {
  const int prec = prec_code<R>();
  const MixShape s = shape(ax.mix, prec, ncols, ncols * nslabs, 32 / (int)sizeof(cplx<R>),
                           128 / (int)sizeof(cplx<R>));
  const int B = s.G * s.ng;
  auto kern = mix_prime_pass(ax.mix) ? k_mcols<DIR, R, true> : k_mcols<DIR, R, false>;
  static bool attr[2] = {false, false};
  FF_TRY(mix_lds_attr(kern, &attr[mix_prime_pass(ax.mix)]));
  // Slabs of fewer than eight workgroups go in order: as ranges, the first of
  // each slab would all run on the first XCD (block b runs on XCD b % 8) and
  // the rest of the eight would be empty.  16 x 16 x 2048 mul!, one workgroup a
  // slab (and no wider than the slab, see shape()): FP32 complex 40 -> 21 us,
  // 4096 fields of 16 x 16 FP64 complex 68 -> 22 us.
  const int64_t wgs = (ncols + B - 1) / B;
  const int64_t per_xcd = nslabs > 1 && wgs < 8 ? 0 : (wgs + 7) / 8;
  const int64_t gx = per_xcd ? 8 * per_xcd : wgs;
  prof_launch("fft_cols_c2c", 2.0 * ncols * nslabs * ax.n * sizeof(cplx<R>), kern,
              dim3((unsigned)gx, (unsigned)nslabs), dim3(mix_wg_threads(ax.mix, B, gx * nslabs)), mix_lds(ax.mix, B, prec),
              st, reinterpret_cast<const cplx<R>*>(in), reinterpret_cast<cplx<R>*>(out), mix_dev(ax.mix, ax.mixtw), ncols, (uint32_t)stride, slab_dist, s, (R)scale, (int)per_xcd);
  FF_LAUNCHED("k_mcols");
  return FFHIP_OK;
}

int mix_rows_c2c(int prec, const void* in, void* out, int64_t nrows, const Axis& ax, int dir, double scale,
                 hipStream_t st) {
  if (prec == FFHIP_F32)
    return dir < 0 ? rows_c2c_t<float, -1>(in, out, nrows, ax, scale, st)
                   : rows_c2c_t<float, 1>(in, out, nrows, ax, scale, st);
  return dir < 0 ? rows_c2c_t<double, -1>(in, out, nrows, ax, scale, st)
                 : rows_c2c_t<double, 1>(in, out, nrows, ax, scale, st);
}

int mix_rows_r2c(int prec, const void* in, void* out, int64_t nrows, const Axis& ax, const void* rtw, hipStream_t st) {
  return prec == FFHIP_F32 ? rows_r2c_t<float>(in, out, nrows, ax, rtw, st)
                           : rows_r2c_t<double>(in, out, nrows, ax, rtw, st);
}

int mix_rows_c2r(int prec, const void* in, void* out, int64_t nrows, const Axis& ax, const void* rtw, double scale,
                 hipStream_t st) {
  return prec == FFHIP_F32 ? rows_c2r_t<float>(in, out, nrows, ax, rtw, scale, st)
                           : rows_c2r_t<double>(in, out, nrows, ax, rtw, scale, st);
}

int mix_cols(int prec, const void* in, void* out, int64_t ncols, int64_t stride, int64_t nslabs, int64_t slab_dist,
             const Axis& ax, int dir, double scale, hipStream_t st) {
  if (prec == FFHIP_F32)
    return dir < 0 ? cols_t<float, -1>(in, out, ncols, stride, nslabs, slab_dist, ax, scale, st)
                   : cols_t<float, 1>(in, out, ncols, stride, nslabs, slab_dist, ax, scale, st);
  return dir < 0 ? cols_t<double, -1>(in, out, ncols, stride, nslabs, slab_dist, ax, scale, st)
                 : cols_t<double, 1>(in, out, ncols, stride, nslabs, slab_dist, ax, scale, st);
}

}  // namespace ffhip
