// Convergence diagnostics of a finished run: cross-chain effective sample
// size and (split) R-hat of draws [n, chains, dims] in float32 or float64,
// computed in float64 (mcmc/diagnostic.py:38-568, stats/sample_stats.py:
// 44-216).
//
// The effective sample size needs, per dimension, the autocovariance at
// every lag averaged over the chains:
//   ess_transpose  draws -> one contiguous row per (dimension, chain)
//   ess_power      per (dimension, block of chains): chains are centred and
//                  transformed two at a time, z = x1 + i x2, zero-padded to
//                  m = 2^ceil(log2 2n) points in LDS, and |Z|^2 is added up.
//                  The real part of the inverse transform of |Z|^2 is the sum
//                  of the two autocorrelations, so neither the two spectra
//                  nor the bit-reversed order of the in-place transform ever
//                  have to be taken apart.
//   ess_finish     per dimension: one inverse transform of the chains' summed
//                  power, the variance of the chain means, the
//                  autocorrelation, its truncation and the sum.
// As float64 library operations (two transforms of every series, complex
// products, copies, a cumulative sum: some forty passes over 65 to 270 MB at
// 1000 x 64 x 127 float32 draws) ESS and split R-hat took 1446 us together;
// these kernels take 81 (each alone: ess_power 36, ess_transpose 20 at 3.3
// TB/s, ess_finish 13, rhat_moments 10, rhat_finish 7; a launch starts under
// the end of the one before).
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "../../include/hipmc.h"
#include "common.h"
#include "runtime.h"

namespace hipmc {
namespace {

struct Cplx {
  double re, im;
};
__device__ inline Cplx operator+(Cplx a, Cplx b) {
  return Cplx{a.re + b.re, a.im + b.im};
}
__device__ inline Cplx operator-(Cplx a, Cplx b) {
  return Cplx{a.re - b.re, a.im - b.im};
}
__device__ inline Cplx operator*(Cplx a, Cplx b) {
  return Cplx{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
// a times -i (forward) or i (inverse)
template <bool INV>
__device__ inline Cplx quarter(Cplx a) {
  return INV ? Cplx{-a.im, a.re} : Cplx{a.im, -a.re};
}

// Unnormalised transforms of 2, 4 and 8 points, results in natural order.
__device__ inline void dft2(Cplx& a, Cplx& b) {
  const Cplx s = a + b;
  b = a - b;
  a = s;
}
template <bool INV>
__device__ inline void dft4(Cplx& a, Cplx& b, Cplx& c, Cplx& d) {
  const Cplx t0 = a + c, t1 = a - c, t2 = b + d, t3 = quarter<INV>(b - d);
  a = t0 + t2;
  c = t0 - t2;
  b = t1 + t3;
  d = t1 - t3;
}
template <bool INV>
__device__ inline void dft8(Cplx (&v)[8]) {
  dft4<INV>(v[0], v[2], v[4], v[6]);  // even terms, results in 0 2 4 6
  dft4<INV>(v[1], v[3], v[5], v[7]);  // odd terms, results in 1 3 5 7
  const double h = 0.70710678118654752440;
  const double s = INV ? h : -h;
  v[3] = v[3] * Cplx{h, s};
  v[5] = quarter<INV>(v[5]);
  v[7] = v[7] * Cplx{-h, s};
  const Cplx e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  const Cplx o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  v[0] = e0 + o0;
  v[1] = e1 + o1;
  v[2] = e2 + o2;
  v[3] = e3 + o3;
  v[4] = e0 - o0;
  v[5] = e1 - o1;
  v[6] = e2 - o2;
  v[7] = e3 - o3;
}

// In-place transform of m = 2^L points by m / 8 threads, one radix-8
// butterfly each per pass: L / 3 radix-8 passes (decimation in frequency),
// the last of which, or the remaining one or two levels, works on the
// thread's eight consecutive points.  Pass i takes blocks of m / 8^i points.
template <int L>
struct Fft {
  static constexpr int M = 1 << L;
  static constexpr int kLive = M / 8;                    // threads with work
  static constexpr int kThreads = kLive < 64 ? 64 : kLive;
  static constexpr int kPasses = (L - 1) / 3;            // twiddled passes
  static constexpr int kLast = L - 3 * kPasses;          // levels of the last
  // One unused element after every eight keeps the last pass (eight
  // consecutive points a thread) and the passes of short blocks off each
  // other's LDS banks.
  static constexpr int kElems = M + M / 8;
  static constexpr size_t kBytes = 2 * (size_t)kElems * sizeof(double);
  static __device__ int at(int i) { return i + (i >> 3); }
  // points of one eighth of a block of pass p
  static constexpr int eighth(int p) { return M >> (3 * (p + 1)); }

  // exp(-2 pi i r / block) of this thread's butterfly in every pass
  static __device__ void twiddles(int tid, Cplx (&w)[kPasses]) {
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int q = eighth(p);
      const int r = tid & (q - 1);
      double s, c;
      sincospi(-2.0 * (double)r / (double)(8 * q), &s, &c);
      w[p] = Cplx{c, s};
    }
  }
  static __device__ int base(int tid, int p) {
    const int q = eighth(p);
    return (tid & ~(q - 1)) * 8 + (tid & (q - 1));
  }
  // v[u] *= w^u (forward) or conj(w)^u (inverse)
  template <bool INV>
  static __device__ void turn(Cplx (&v)[8], Cplx w) {
    if (INV) w.im = -w.im;
    const Cplx w2 = w * w, w3 = w2 * w, w4 = w2 * w2;
    v[1] = v[1] * w;
    v[2] = v[2] * w2;
    v[3] = v[3] * w3;
    v[4] = v[4] * w4;
    v[5] = v[5] * (w4 * w);
    v[6] = v[6] * (w4 * w2);
    v[7] = v[7] * (w4 * w3);
  }
  template <bool INV>
  static __device__ void last(Cplx (&v)[8]) {
    if (kLast == 1) {
#pragma unroll
      for (int u = 0; u < 8; u += 2) dft2(v[u], v[u + 1]);
    } else if (kLast == 2) {
#pragma unroll
      for (int u = 0; u < 8; u += 4)
        dft4<INV>(v[u], v[u + 1], v[u + 2], v[u + 3]);
    } else {
      dft8<INV>(v);
    }
  }
  static __device__ void put(double* re, double* im, int i0, int step,
                             const Cplx (&v)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = at(i0 + u * step);
      re[k] = v[u].re;
      im[k] = v[u].im;
    }
  }
  static __device__ void get(const double* re, const double* im, int i0,
                             int step, Cplx (&v)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = at(i0 + u * step);
      v[u] = Cplx{re[k], im[k]};
    }
  }
  // v: points tid + u * M / 8 on entry; on return the thread's eight
  // consecutive results of the transform's own order.  Every thread of the
  // block calls it (it holds barriers); threads past kLive do no work.
  static __device__ void forward(double* re, double* im, int tid,
                                 const Cplx (&w)[kPasses], Cplx (&v)[8]) {
    const bool live = tid < kLive;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      if (live) {
        if (p > 0) get(re, im, base(tid, p), eighth(p), v);
        dft8<false>(v);
        turn<false>(v, w[p]);
        put(re, im, base(tid, p), eighth(p), v);
      }
      __syncthreads();
    }
    if (live) {
      get(re, im, 8 * tid, 1, v);
      last<false>(v);
    }
  }
  // The inverse of forward() times M.
  static __device__ void inverse(double* re, double* im, int tid,
                                 const Cplx (&w)[kPasses], Cplx (&v)[8]) {
    const bool live = tid < kLive;
    if (live) {
      last<true>(v);
      put(re, im, 8 * tid, 1, v);
    }
    __syncthreads();
#pragma unroll
    for (int p = kPasses - 1; p >= 0; --p) {
      if (live) {
        get(re, im, base(tid, p), eighth(p), v);
        turn<true>(v, w[p]);
        dft8<true>(v);
        if (p > 0) put(re, im, base(tid, p), eighth(p), v);
      }
      __syncthreads();
    }
  }
};

// Sum over the block's threads of a and b, given to every thread; `red` holds
// 2 doubles per wave.  Ends with the buffer free for the next call.
__device__ inline void block_sum2(double& a, double& b, double* red) {
  const int wave = threadIdx.x >> 6, waves = (blockDim.x + 63) >> 6;
  double sa, sb;
  wave_sum2(a, b, sa, sb);
  if (lane_id() == 0) {
    red[2 * wave] = sa;
    red[2 * wave + 1] = sb;
  }
  __syncthreads();
  a = 0.0;
  b = 0.0;
  for (int w = 0; w < waves; ++w) {
    a += red[2 * w];
    b += red[2 * w + 1];
  }
  __syncthreads();
}

// draws x[t * sn + c * sc + d * sd] -> out[(d * chains + c) * n + t].  Tiles of
// 64 draws x 64 series (series s = c * dims + d, so that consecutive lanes
// read consecutive dimensions) turned over in LDS.
template <typename T>
__global__ void __launch_bounds__(256)
    ess_transpose(const T* __restrict__ x, int n, int chains, int dims,
                  int64_t sn, int64_t sc, int64_t sd, T* __restrict__ out) {
  __shared__ T tile[64][65];
  const int64_t series = (int64_t)chains * dims;
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int64_t s0 = (int64_t)blockIdx.x * 64;
  const int t0 = blockIdx.y * 64;
  {
    const int64_t s = s0 + lane;
    if (s < series) {
      const int64_t c = s / dims, d = s - c * dims;
      const T* src = x + c * sc + d * sd;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = t0 + part + 4 * i;
        if (t < n) tile[part + 4 * i][lane] = src[(int64_t)t * sn];
      }
    }
  }
  __syncthreads();
  const int t = t0 + lane;
  if (t >= n) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t s = s0 + part + 4 * i;
    if (s >= series) return;
    const int64_t c = s / dims, d = s - c * dims;
    out[(d * chains + c) * n + t] = tile[lane][part + 4 * i];
  }
}

// Block (d, y): chain pairs [y * per, (y + 1) * per) of dimension d.  Writes
// the chains' means [dims, chains] and this block's summed power
// [blocks y, dims, m].
// Bound by the serial passes of a pair (four at 2048 points, 192 KiB through
// LDS) at two blocks a CU: the butterflies take 189 registers; held to 168 for
// three blocks a CU they spill, 36 -> 43 us at 1000 x 64 x 127.
template <typename T, int L>
__global__ void __launch_bounds__(Fft<L>::kThreads)
    ess_power(const T* __restrict__ rows, int n, int chains, int dims, int per,
              double* __restrict__ means, double* __restrict__ power) {
  using F = Fft<L>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double red[2 * (F::kThreads / 64)];
  double* re = (double*)smem_raw;
  double* im = re + F::kElems;
  const int tid = threadIdx.x;
  const int d = blockIdx.x;
  Cplx w[F::kPasses];
  F::twiddles(tid, w);
  double acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = 0.0;
  const int pairs = (chains + 1) >> 1;
  const int p1 = min(pairs, (int)(blockIdx.y + 1) * per);
  // the thread's draws of a pair (t = tid + u m / 8; n <= m / 2): the next
  // pair's are loaded while the current one is transformed
  T a1[4], a2[4];
  auto load = [&](int p) {
    const int c = 2 * p;
    const T* x1 = rows + ((size_t)d * chains + c) * n;
    const T* x2 = c + 1 < chains ? x1 + n : x1;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = tid + u * (F::M / 8);
      const bool in = tid < F::kLive && t < n;
      a1[u] = in ? x1[t] : T(0);
      a2[u] = in ? x2[t] : T(0);
    }
  };
  const int p0 = blockIdx.y * per;
  if (p0 < p1) load(p0);
  for (int p = p0; p < p1; ++p) {
    const int c = 2 * p;
    const bool two = c + 1 < chains;
    double m1 = 0.0, m2 = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      m1 += (double)a1[u];
      m2 += (double)a2[u];
    }
    block_sum2(m1, m2, red);
    m1 /= (double)n;
    m2 /= (double)n;
    if (tid == 0) {
      means[(size_t)d * chains + c] = m1;
      if (two) means[(size_t)d * chains + c + 1] = m2;
    }
    Cplx v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = tid + u * (F::M / 8);
      const bool in = tid < F::kLive && u < 4 && t < n;
      v[u].re = in ? (double)a1[u & 3] - m1 : 0.0;
      v[u].im = in && two ? (double)a2[u & 3] - m2 : 0.0;
    }
    if (p + 1 < p1) load(p + 1);
    F::forward(re, im, tid, w, v);
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] += v[u].re * v[u].re + v[u].im * v[u].im;
    __syncthreads();  // the next pair overwrites the buffer
  }
  if (tid < F::kLive) {
    double* out = power + ((size_t)blockIdx.y * dims + d) * F::M + tid;
#pragma unroll
    for (int u = 0; u < 8; ++u) out[u * F::kLive] = acc[u];
  }
}

// One block per dimension.  With ac[k] the mean over the chains of the
// autocovariance at lag k, w = ac[0] and b the variance of the chain means:
//   rho[k] = 1 - (w - ac[k]) / (w + b),
//   ess = chains n / (-1 + 2 sum_k (n - k) / n rho[k] keep[k])
// where keep is 1 before the first rho below `threshold` and 0 from it on
// (always 1 if truncate is 0).  The terms are multiplied by keep, so a NaN
// beyond the truncation makes the result NaN as it does in the reference.
template <int L>
__global__ void __launch_bounds__(Fft<L>::kThreads)
    ess_finish(const double* __restrict__ power, int blocks, int n, int chains,
               int dims, const double* __restrict__ means, int truncate,
               double threshold, double* __restrict__ out) {
  using F = Fft<L>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double red[2 * (F::kThreads / 64)];
  __shared__ double lag0;
  __shared__ int first;
  double* re = (double*)smem_raw;
  double* im = re + F::kElems;
  const int tid = threadIdx.x;
  const int d = blockIdx.x;
  Cplx w[F::kPasses];
  F::twiddles(tid, w);
  Cplx v[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = Cplx{0.0, 0.0};
  if (tid < F::kLive) {
#pragma unroll 4
    for (int y = 0; y < blocks; ++y) {
      const double* src = power + ((size_t)y * dims + d) * F::M + tid;
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u].re += src[u * F::kLive];
    }
  }
  if (tid == 0) first = n;
  F::inverse(re, im, tid, w, v);
  // v[u].re = M chains (n - k) ac[k] at k = tid + u M / 8
  double ac[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int k = tid + u * (F::M / 8);
    ac[u] = k < n ? v[u].re / ((double)F::M * (double)chains * (double)(n - k))
                  : 0.0;
  }
  if (tid == 0) lag0 = ac[0];
  double s = 0.0, q = 0.0;
  for (int c = tid; c < chains; c += F::kThreads)
    s += means[(size_t)d * chains + c];
  block_sum2(s, q, red);  // its barriers also publish lag0 and first
  const double mu = s / (double)chains;
  s = 0.0;
  for (int c = tid; c < chains; c += F::kThreads) {
    const double e = means[(size_t)d * chains + c] - mu;
    s += e * e;
  }
  block_sum2(s, q, red);
  const double var = s / (double)(chains - 1);
  const double w0 = lag0;
  double rho[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int k = tid + u * (F::M / 8);
    rho[u] = 1.0 - (w0 - ac[u]) / (w0 + var);
    if (truncate && tid < F::kLive && k < n && rho[u] < threshold)
      atomicMin(&first, k);
  }
  __syncthreads();
  double total = 0.0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int k = tid + u * (F::M / 8);
    if (tid < F::kLive && k < n)
      total += (double)(n - k) / (double)n * rho[u] * (k < first ? 1.0 : 0.0);
  }
  double none = 0.0;
  block_sum2(total, none, red);
  if (tid == 0)
    out[d] = (double)chains * (double)n / (-1.0 + 2.0 * total);
}

// Count, mean and sum of squared deviations from the mean of some draws.
struct Moments {
  double n, mean, m2;
};
// Those of both sets together (either may be empty).  Equal means stay as they
// are, so that the variance of equal draws is zero.
__device__ inline Moments merge(const Moments& a, const Moments& b) {
  const double n = a.n + b.n, r = b.n / n, d = b.mean - a.mean;
  const Moments m{n, a.mean + d * r, (a.m2 + b.m2) + d * (d * (a.n * r))};
  return b.n == 0.0 ? a : (a.n == 0.0 ? b : m);
}

// Mean and sum of squared deviations of every series (and half of it, with
// halves = 2) over one time chunk: groups of kGroup draws by two passes in
// registers (about their first draw, then about their mean), groups and threads
// merged.  No pivot is common to more than a group, so an outlier costs the
// other draws no precision: split R-hat of 4 chains of 20000 draws, whose first
// is 100 standard deviations out, is off by 4e-16 (sums about the first draw:
// 4e-12).
// Block: 2^width_log adjacent series x its other threads in time steps, grid y
// = half, z = time chunk; out [z, half, 2, series].  Bound by HBM (each draw is
// read once).
template <typename T>
__global__ void __launch_bounds__(256)
    rhat_moments(const T* __restrict__ x, int h, int chains, int dims,
                 int64_t sn, int64_t sc, int64_t sd, int chunk, int width_log,
                 double* __restrict__ out) {
  constexpr int kGroup = 16;
  __shared__ double red[3][256];
  const int tid = threadIdx.x;
  const int lane = tid & ((1 << width_log) - 1), part = tid >> width_log;
  const int parts = 256 >> width_log;
  const int64_t series = (int64_t)chains * dims;
  const int64_t s = ((int64_t)blockIdx.x << width_log) + lane;
  Moments m{0.0, 0.0, 0.0};
  if (s < series) {
    const int64_t c = s / dims, d = s - c * dims;
    const T* src = x + c * sc + d * sd + (int64_t)blockIdx.y * h * sn;
    const int64_t t0 = (int64_t)blockIdx.z * chunk;
    const int t1 = (int)(t0 + chunk < h ? t0 + chunk : h);
    for (int64_t t = t0 + part; t < t1; t += kGroup * parts) {
      T v[kGroup];
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        const int64_t tu = t + (int64_t)u * parts;
        v[u] = src[(tu < t1 ? tu : t1 - 1) * sn];
      }
      const int64_t left = (t1 - t + parts - 1) / parts;
      const int live = left < kGroup ? (int)left : kGroup;
      const double x0 = (double)v[0];
      double e[kGroup], sum = 0.0;
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        e[u] = (double)v[u] - x0;
        sum += u < live ? e[u] : 0.0;
      }
      const double mean = sum / (double)live;
      double m2 = 0.0;
#pragma unroll
      for (int u = 0; u < kGroup; ++u)
        m2 += u < live ? (e[u] - mean) * (e[u] - mean) : 0.0;
      m = merge(m, Moments{(double)live, x0 + mean, m2});
    }
  }
  red[0][tid] = m.n;
  red[1][tid] = m.mean;
  red[2][tid] = m.m2;
  for (int k = 128; k >= 1 << width_log; k >>= 1) {
    __syncthreads();
    if (tid < k) {
      m = merge(m, Moments{red[0][tid + k], red[1][tid + k], red[2][tid + k]});
      red[0][tid] = m.n;
      red[1][tid] = m.mean;
      red[2][tid] = m.m2;
    }
  }
  if (part == 0 && s < series) {
    double* o = out + ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * 2 * series;
    o[s] = m.mean;
    o[series + s] = m.m2;
  }
}

// How rhat_finish shares a dimension's m series out.
struct RhatShare {
  int threads;    // of a block
  int share_log;  // log2 of a block's threads on one dimension
  int splits;     // blocks on one dimension
};

__device__ inline double rhat_of(const Moments& means, double var, int m,
                                 double h) {
  const double w = var / (double)m;
  const double s2 = (h - 1.0) / h * w + means.m2 / ((double)m - 1.0);
  return ((double)m + 1.0) / (double)m * s2 / w - (h - 1.0) / ((double)m * h);
}

// With the mean and unbiased variance of each of a dimension's m = halves *
// chains series of h draws, w the mean of the variances and b the unbiased
// variance of the means,
//   s2 = (h - 1) / h w + b,  R-hat = (m + 1) / m s2 / w - (h - 1) / (m h).
// Block (adjacent dimensions, range of series).  With several ranges a block
// leaves its sums in place of its range's first two series (no other block
// reads them) for rhat_combine.
__global__ void __launch_bounds__(1024)
    rhat_finish(double* sums, int h, int halves, int chains, int dims,
                int chunk, int chunks, RhatShare share,
                double* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* red = (double*)smem_raw;  // 4 x threads
  const int tid = threadIdx.x, nt = blockDim.x;
  const int width = nt >> share.share_log;
  const int part = tid / width, parts = 1 << share.share_log;
  const int64_t d = (int64_t)blockIdx.x * width + (tid - part * width);
  const int64_t series = (int64_t)chains * dims;
  const int m = halves * chains;
  const int per = (m + share.splits - 1) / share.splits;
  const int i0 = blockIdx.y * per, i1 = min(m, i0 + per);
  const double hn = (double)h;
  auto row = [&](int i) {  // of chunk 0
    const int half = i / chains, c = i - half * chains;
    return sums + (size_t)half * 2 * series + (int64_t)c * dims + d;
  };
  Moments means{0.0, 0.0, 0.0};
  double var = 0.0;
  if (d < dims) {
    if (chunks == 1) {
#pragma unroll 8
      for (int i = i0 + part; i < i1; i += parts) {
        const double* p = row(i);
        var += p[series] / (hn - 1.0);
        means = merge(means, Moments{1.0, p[0], 0.0});
      }
    } else {
      for (int i = i0 + part; i < i1; i += parts) {
        const double* p = row(i);
        Moments a{0.0, 0.0, 0.0};
#pragma unroll 8
        for (int z = 0; z < chunks; ++z, p += (size_t)halves * 2 * series) {
          const int n = min(chunk, h - z * chunk);
          a = merge(a, Moments{(double)(n > 0 ? n : 0), p[0], p[series]});
        }
        var += a.m2 / (hn - 1.0);
        means = merge(means, Moments{1.0, a.mean, 0.0});
      }
    }
  }
  for (int k = nt >> 1; k >= width; k >>= 1) {
    red[tid] = means.n;
    red[nt + tid] = means.mean;
    red[2 * nt + tid] = means.m2;
    red[3 * nt + tid] = var;
    __syncthreads();
    if (tid < k) {
      const int o = tid + k;
      means = merge(means, Moments{red[o], red[nt + o], red[2 * nt + o]});
      var += red[3 * nt + o];
    }
    __syncthreads();
  }
  if (part != 0 || d >= dims) return;
  if (share.splits == 1) {
    out[d] = rhat_of(means, var, m, hn);
  } else {
    double* p = row(i0);
    p[0] = means.mean;
    p[series] = means.m2;
    row(i0 + 1)[0] = var;
  }
}

// One thread per dimension: the ranges of rhat_finish in order.
__global__ void __launch_bounds__(256)
    rhat_combine(const double* __restrict__ sums, int h, int halves, int chains,
                 int dims, int splits, double* __restrict__ out) {
  const int64_t d = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (d >= dims) return;
  const int64_t series = (int64_t)chains * dims;
  const int m = halves * chains;
  const int per = (m + splits - 1) / splits;
  auto row = [&](int i) {
    const int half = i / chains, c = i - half * chains;
    return sums + (size_t)half * 2 * series + (int64_t)c * dims + d;
  };
  Moments means{0.0, 0.0, 0.0};
  double var = 0.0;
#pragma unroll 8
  for (int y = 0; y < splits; ++y) {
    const int i0 = y * per;
    const double* p = row(i0);
    means = merge(means,
                  Moments{(double)(min(m, i0 + per) - i0), p[0], p[series]});
    var += row(i0 + 1)[0];
  }
  out[d] = rhat_of(means, var, m, (double)h);
}

// One thread per series, up to a block of adjacent dimensions, but fewer (down
// to one per eight series) where the dimensions alone fill the GPU; several
// blocks where a dimension has thousands of series.  Each range has at least
// two series.  Split R-hat, us, torch form / one block of 256 threads per
// dimension, whatever its series / now: 65 draws, 2 chains, 1e6 dimensions 881 /
// 1642 / 230; 65 draws, 250000 chains, 1 dimension 128 / 354 / 62; 1000 draws,
// 100000 chains, 1 dimension 684 / 762 / 111.
RhatShare rhat_share(int m, int dims) {
  int log = 0;
  while (log < 10 && (1 << log) < m) ++log;
  while (log > 0 && ((int64_t)dims << log) > (1 << 17) && m < (8 << log)) --log;
  if (log <= 8) return RhatShare{256, log, 1};
  for (int w = 1; w < 8 && w < dims; w <<= 1) --log;
  int splits = 1;
  while (splits < 32 && m >= (2 << log) * 2 * splits &&
         ((int64_t)dims << log) * splits < (1 << 17))
    splits <<= 1;
  return RhatShare{1024, log, splits};
}

template <typename F>
int allow_dynamic_lds(F* kernel, size_t bytes) {
  if (bytes <= (size_t)kMaxLdsPerBlock) return HIPMC_OK;
  return hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)bytes),
                   "hipFuncSetAttribute(max dynamic LDS)");
}

template <typename T, int L>
int ess_launch(const T* rows, int n, int chains, int dims, int blocks,
               int truncate, double threshold, double* means, double* power,
               double* out, hipStream_t s) {
  using F = Fft<L>;
  int rc = allow_dynamic_lds(&ess_power<T, L>, F::kBytes);
  if (rc != HIPMC_OK) return rc;
  rc = allow_dynamic_lds(&ess_finish<L>, F::kBytes);
  if (rc != HIPMC_OK) return rc;
  const int pairs = (chains + 1) / 2;
  const int per = (pairs + blocks - 1) / blocks;
  hipLaunchKernelGGL((ess_power<T, L>), dim3(dims, blocks), dim3(F::kThreads),
                     F::kBytes, s, rows, n, chains, dims, per, means, power);
  hipLaunchKernelGGL((ess_finish<L>), dim3(dims), dim3(F::kThreads), F::kBytes,
                     s, power, blocks, n, chains, dims, means, truncate,
                     threshold, out);
  return hip_check(hipGetLastError(), "ess launch");
}

template <typename T>
int ess_run(int n, int chains, int dims, int64_t sn, int64_t sc, int64_t sd,
            const T* x, int truncate, double threshold, int blocks, T* rows,
            double* means, double* power, double* out, hipStream_t s) {
  const int64_t series = (int64_t)chains * dims;
  hipLaunchKernelGGL(ess_transpose<T>,
                     dim3((unsigned)((series + 63) / 64), (n + 63) / 64),
                     dim3(256), 0, s, x, n, chains, dims, sn, sc, sd, rows);
  int l = 4;
  while ((1 << l) < 2 * n) ++l;
  switch (l) {
#define HIPMC_ESS(LL)                                                       \
  case LL:                                                                  \
    return ess_launch<T, LL>(rows, n, chains, dims, blocks, truncate,       \
                             threshold, means, power, out, s);
    HIPMC_ESS(4) HIPMC_ESS(5) HIPMC_ESS(6) HIPMC_ESS(7) HIPMC_ESS(8)
    HIPMC_ESS(9) HIPMC_ESS(10) HIPMC_ESS(11) HIPMC_ESS(12) HIPMC_ESS(13)
#undef HIPMC_ESS
  }
  return fail(HIPMC_E_UNSUPPORTED, "ess: more than 4096 draws");
}

template <typename T>
int rhat_run(int h, int halves, int chains, int dims, int64_t sn, int64_t sc,
             int64_t sd, const T* x, int chunks, double* sums, double* out,
             hipStream_t s) {
  const int64_t series = (int64_t)chains * dims;
  const int chunk = (h + chunks - 1) / chunks;
  int w = 0;  // adjacent series of a block: as many as there are, at most 64
  while (w < 6 && ((int64_t)1 << w) < series) ++w;
  hipLaunchKernelGGL(rhat_moments<T>,
                     dim3((unsigned)((series + (1 << w) - 1) >> w), halves,
                          chunks),
                     dim3(256), 0, s, x, h, chains, dims, sn, sc, sd, chunk, w,
                     sums);
  const RhatShare share = rhat_share(halves * chains, dims);
  const int width = share.threads >> share.share_log;
  hipLaunchKernelGGL(rhat_finish,
                     dim3((dims + width - 1) / width, share.splits),
                     dim3(share.threads), 4 * share.threads * sizeof(double),
                     s, sums, h, halves, chains, dims, chunk, chunks, share,
                     out);
  if (share.splits > 1)
    hipLaunchKernelGGL(rhat_combine, dim3((dims + 255) / 256), dim3(256), 0, s,
                       sums, h, halves, chains, dims, share.splits, out);
  return hip_check(hipGetLastError(), "rhat launch");
}

int check_draws(const char* what, int32_t dtype, int64_t n, int64_t chains,
                int64_t dims) {
  if (dtype != HIPMC_F32 && dtype != HIPMC_F64)
    return fail(HIPMC_E_INVALID, std::string(what) + ": bad dtype");
  if (n < 1 || chains < 1 || dims < 1)
    return fail(HIPMC_E_INVALID,
                std::string(what) + ": draws, chains and dims must be >= 1");
  if (chains > (1 << 30) || dims > (1 << 30) || chains * dims > (1LL << 36))
    return fail(HIPMC_E_UNSUPPORTED, std::string(what) + ": too many series");
  return HIPMC_OK;
}

}  // namespace
}  // namespace hipmc

using namespace hipmc;

extern "C" {

int hipmc_effective_sample_size(int32_t dtype, int64_t n, int64_t chains,
                                int64_t dims, int64_t stride_n,
                                int64_t stride_chain, int64_t stride_dim,
                                const void* x, int32_t truncate,
                                double threshold, int32_t blocks, void* ws_rows,
                                double* ws_means, double* ws_power, double* out,
                                uint64_t stream) {
  const int rc = check_draws("ess", dtype, n, chains, dims);
  if (rc) return rc;
  if (!x || !ws_rows || !ws_means || !ws_power || !out)
    return fail(HIPMC_E_INVALID, "ess: NULL argument");
  if (chains < 2) return fail(HIPMC_E_INVALID, "ess: needs > 1 chain");
  if (n > 4096) return fail(HIPMC_E_UNSUPPORTED, "ess: more than 4096 draws");
  if (blocks < 1 || blocks > 65535)
    return fail(HIPMC_E_INVALID, "ess: blocks must be in [1, 65535]");
  hipStream_t s = as_stream(stream);
  if (dtype == HIPMC_F32)
    return ess_run((int)n, (int)chains, (int)dims, stride_n, stride_chain,
                   stride_dim, (const float*)x, truncate, threshold, blocks,
                   (float*)ws_rows, ws_means, ws_power, out, s);
  return ess_run((int)n, (int)chains, (int)dims, stride_n, stride_chain,
                 stride_dim, (const double*)x, truncate, threshold, blocks,
                 (double*)ws_rows, ws_means, ws_power, out, s);
}

int hipmc_potential_scale_reduction(int32_t dtype, int64_t n, int64_t chains,
                                    int64_t dims, int64_t stride_n,
                                    int64_t stride_chain, int64_t stride_dim,
                                    const void* x, int32_t split,
                                    int32_t chunks, double* ws_sums,
                                    double* out, uint64_t stream) {
  const int rc = check_draws("rhat", dtype, n, chains, dims);
  if (rc) return rc;
  if (!x || !ws_sums || !out)
    return fail(HIPMC_E_INVALID, "rhat: NULL argument");
  const int halves = split ? 2 : 1;
  if (n / halves < 2 || n > (1 << 30))
    return fail(HIPMC_E_INVALID, "rhat: needs 2 to 2^30 draws per half");
  if (chains > (1 << 29))
    return fail(HIPMC_E_UNSUPPORTED, "rhat: too many chains");
  if (chunks < 1 || chunks > 65535)
    return fail(HIPMC_E_INVALID, "rhat: chunks must be in [1, 65535]");
  // a grid holds fewer than 2^32 threads: 256 per 64 series
  if (chains * dims >= 1 << 30)
    return fail(HIPMC_E_UNSUPPORTED, "rhat: too many series");
  const int h = (int)(n / halves);
  hipStream_t s = as_stream(stream);
  if (dtype == HIPMC_F32)
    return rhat_run(h, halves, (int)chains, (int)dims, stride_n, stride_chain,
                    stride_dim, (const float*)x, chunks, ws_sums, out, s);
  return rhat_run(h, halves, (int)chains, (int)dims, stride_n, stride_chain,
                  stride_dim, (const double*)x, chunks, ws_sums, out, s);
}

}  // extern "C"
