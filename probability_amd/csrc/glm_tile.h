// GLM log densities and gradients of many chains on matrix instructions.
//
// A launch whose chains share a design matrix X [n, dx] is two products, the
// logits X B (B the chains' coefficients, one column a chain) and the
// gradients R^T X (R the residuals), both with as many columns as chains:
// v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64 work in the state's own
// precision.  The sampling kernels' per-chain passes (targets.h) leave the
// matrix cores idle and read X once per chain; these read it once per 16 or 32
// chains, and split the rows over blocks so that a few tiles of chains still
// fill the chip.
//   glm_tile_grad    one block per (tile of chains, range of rows): partial
//                    gradients and log-likelihoods (or residual sums of
//                    squares) to a workspace
//   glm_tile_finish  one wave (or block) per chain: adds the ranges in order,
//                    prior and bijector terms (log density and gradient out)
//   glm_tile_step    one wave (or block) per chain: the same sums, then the
//                    leapfrog / Metropolis-Hastings arithmetic of hmc_kernel
// Log density and gradient, us, one chain per wave -> tiled (float32): 2048 x
// 64, 1024 chains 39 -> 18; 6001 x 101, 512 chains 161 -> 29; 8192 x 128, 32
// chains 211 -> 16; 8192 x 128, 2048 chains 305 -> 106 (81 TFLOP/s of 150 that
// a large float32 matrix product reaches); float64 8000 x 127, 1000 chains 681
// -> 140.  Large launches are bound by the matrix instructions and the
// sigmoids between them, which overlap little (matrix cores busy for half of
// the largest, a third of 6001 x 101, 512 chains); small ones by the two
// launches and their blocks' fixed part, some 9 us.
#pragma once

#include "../../include/hipmc.h"
#include "common.h"
#include "kernels.h"
#include "runtime.h"
#include "targets.h"

namespace hipmc {

template <typename T>
struct Quad {
  typedef T type __attribute__((ext_vector_type(4)));
};

// D += A B with A 16 x 4, B 4 x 16: lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16], and register i of the result is row tile_row<T>(i, l / 16),
// column l % 16.
__device__ inline Quad<float>::type mfma16x4(float a, float b,
                                             Quad<float>::type c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ inline Quad<double>::type mfma16x4(double a, double b,
                                              Quad<double>::type c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <typename T>
__device__ inline int tile_row(int i, int g) {
  return sizeof(T) == 4 ? 4 * g + i : 4 * i + g;
}

__device__ inline GlmTile glm_tile_of(const GlmTileArgs& a, int tile, int ct) {
  if (a.tiles) return a.tiles[tile];
  GlmTile t;
  t.prob = 0;
  t.chain0 = tile * ct;
  t.n_chains = a.n_chains - t.chain0 < ct ? a.n_chains - t.chain0 : ct;
  t.n_split = a.n_split;
  t.slot0 = tile * a.n_split;
  t.rows = a.rows;
  return t;
}

// LDS pitch of a staged row of 16 S elements: the 16-byte row writes of eight
// consecutive lanes and the column reads of a wave fall in distinct banks.
template <typename T>
__host__ __device__ constexpr int tile_pitch(int s) {
  return 16 * s + (sizeof(T) == 4 ? 4 : 2);
}
// LDS of a block: the waves' staged rows, reused for their partial gradients
// at the end, and their partial sums.
template <typename T, int NG>
__host__ __device__ constexpr size_t glm_tile_sums_at(int s) {
  const size_t rows = 16 * (size_t)tile_pitch<T>(s), part = 256 * (size_t)NG * s;
  return sizeof(T) * kTileWaves * (rows > part ? rows : part);
}
template <typename T, int NG>
__host__ __device__ constexpr size_t glm_tile_lds(int s) {
  return glm_tile_sums_at<T, NG>(s) + sizeof(double) * kTileWaves * NG * 16;
}

// The rows [row0, row1) of X for NG groups of 16 chains, coefficients in S
// slabs of 16.  Wave w takes sub-tiles of 16 rows 64 apart.  Lane (m = l % 16,
// g = l / 16):
//  loads   row m, coefficients 16 s + 4 g + [0, 4) (16 bytes a slab, 64
//          contiguous bytes of a row over its four lanes), also written to the
//          wave's LDS rows;
//  logits  step (s, t): A = element t of the loaded slab (k = 16 s + 4 g + t),
//          B = the same coefficient of chain m; lane (m, g) ends with rows
//          tile_row(i, g) of chain m;
//  gradient step (s, i): A = residual i (chain m, row tile_row(i, g)), B = X at
//          that row, coefficient 16 s + m, read back from LDS; lane (m, g)
//          accumulates chains tile_row(i, g) of coefficient 16 s + m.
// The next rows' loads are in flight during the residuals and the gradient.
// Rows past row1 read a row inside and get residual zero; coefficients past dx
// are zero in B, and columns past the row pitch are not read.
template <typename T, int S, int NG>
__device__ __attribute__((always_inline)) inline void glm_tile_rows(
    const hipmc_problem& pb, const GlmTile& tile, const GlmTileArgs& a,
    int row0, int row1, bool want_sum, int slot, unsigned char* smem) {
  using Q = typename Quad<T>::type;
  constexpr int P = tile_pitch<T>(S);
  constexpr int CT = 16 * NG;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, m = l & 15, g = l >> 4;
  const bool linear = pb.kind == HIPMC_TARGET_LINEAR;
  const int dx = linear ? pb.dim - 1 : pb.dim;
  const int xp = pb.x_pitch;
  const gptr<T> X = (gptr<T>)pb.x;
  const gptr<T> Y = (gptr<T>)pb.y;
  lptr<T> rows = (lptr<T>)((T*)smem + (size_t)w * 16 * P);
  // the chains' coefficients, bijectors applied (chains past the tile's and
  // coefficients past dx read one inside and are zero)
  typedef T QU __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  Q beta[NG][S];
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    const int c = 16 * j + m;
    const bool in = c < tile.n_chains;
    const T* q = (const T*)a.x + (size_t)(tile.chain0 + (in ? c : 0)) * a.stride;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (s + 1 < S) {
        beta[j][s] = *(const QU*)(q + 16 * s + 4 * g);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int e = 16 * s + 4 * g + t;
          const T v = q[e < dx ? e : dx - 1];
          beta[j][s][t] = e < dx ? v : T(0);
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) beta[j][s][t] = in ? beta[j][s][t] : T(0);
    }
  }
  for (int r = 0; r < pb.n_bij; ++r) {
    const int b0 = pb.bij_off[r], b1 = b0 + pb.bij_len[r];
    if (b0 >= dx) continue;
#pragma unroll
    for (int j = 0; j < NG; ++j)
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int e = 16 * s + 4 * g + t;
          const T v = beta[j][s][t];
          T f = v;
          if (pb.bij_code[r] == HIPMC_BIJ_SOFTPLUS)
            f = fmax(v, T(0)) + softplus_parts(v).l;
          else if (pb.bij_code[r] == HIPMC_BIJ_EXP)
            f = exp(v);
          beta[j][s][t] = e >= b0 && e < b1 && e < dx ? f : v;
        }
  }
  Q acc[NG][S];
  double sum[NG];
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    sum[j] = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) acc[j][s] = Q{T(0), T(0), T(0), T(0)};
  }
  Q xv[S];
  T yv[4];
  auto load = [&](int r0) {
    const int j = r0 + m;
    const gptr<T> src = X + (size_t)(j < row1 ? j : row1 - 1) * xp + 4 * g;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      // every slab but the last lies inside the row
      if (s + 1 < S || 16 * s + 4 * g < xp)
        xv[s] = *(gptr<Q>)(src + 16 * s);
      else
        xv[s] = Q{T(0), T(0), T(0), T(0)};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + tile_row<T>(i, g);
      yv[i] = Y[r < row1 ? r : row1 - 1];
    }
  };
  int r0 = row0 + 16 * w;
  if (r0 < row1) load(r0);
  for (; r0 < row1; r0 += kTileRows) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      *(lptr<Q>)(rows + m * P + 16 * s + 4 * g) = xv[s];
    // Logits are summed in four parts (each step t apart), or eight (two sets
    // of slabs as well): one chain of additions over all columns doubles their
    // rounding error, and a linear model's residual is a small difference of
    // them.  Relative error of its gradient, float32 at 8192 x 128 against
    // float64: one chain 2.8e-6, four parts 1.5e-6, eight 1.2e-6 (the per-chain
    // pass 1.2e-6); sixteen parts spill (8192 x 128, 2048 chains a third slower).
    // Float64 at 1024 to 1300 rows near the mode, one chain / four / eight
    // parts, rms error against extended precision over the per-chain pass's:
    // 127 columns 1.98 / 1.07 / 0.87, 96 columns 1.50 / 0.89 / 0.75, 64 columns
    // 1.55 / 0.92 / 0.78; so eight from 97 columns on.  (8000 x 127, 1000
    // chains 130 / 131 / 140 us, where eight spill; 4000 x 64, 1000 chains 50 /
    // 49 / 65.)
    constexpr int kSets = S < (sizeof(T) == 4 ? 2 : 7) ? 1 : 2;
    Q lg[NG];
#pragma unroll
    for (int h = 0; h < kSets; ++h) {
      Q part[4][NG];
#pragma unroll
      for (int s = h; s < S; s += kSets)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int j = 0; j < NG; ++j)
            part[t][j] = mfma16x4(
                xv[s][t], beta[j][s][t],
                s == h ? Q{T(0), T(0), T(0), T(0)} : part[t][j]);
#pragma unroll
      for (int j = 0; j < NG; ++j) {
        const Q sum = (part[0][j] + part[1][j]) + (part[2][j] + part[3][j]);
        lg[j] = h == 0 ? sum : lg[j] + sum;
      }
    }
    T yc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) yc[i] = yv[i];
    if (r0 + kTileRows < row1) load(r0 + kTileRows);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // one branch for all of the lane's elements, so that their chains of
    // dependent operations interleave
    T res[NG][4];
    bool valid[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) valid[i] = r0 + tile_row<T>(i, g) < row1;
    if (linear) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NG; ++j) {
          const T r = valid[i] ? yc[i] - lg[j][i] : T(0);
          sum[j] += (double)(r * r);
          res[j][i] = r;
        }
    } else if (want_sum || sizeof(T) == 8) {
      // (float64: the branch below spills, and adds a third to a gradient at
      // 8000 x 127, 1000 chains, more than the log-likelihood it saves)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NG; ++j) {
          const T s = lg[j][i], yy = yc[i], w0 = T(1) - yy;
          const SoftplusParts<T> sp = softplus_parts(s);
          const T l0 = w0 == T(0) ? T(0) : -(fmax(s, T(0)) + sp.l) * w0;
          const T l1 = yy == T(0) ? T(0) : -(fmax(-s, T(0)) + sp.l) * yy;
          sum[j] += valid[i] ? (double)(l0 + l1) : 0.0;
          res[j][i] = valid[i] ? yy - sp.sig : T(0);
        }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NG; ++j)
          res[j][i] = valid[i] ? yc[i] - softplus_parts(lg[j][i]).sig : T(0);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const T xc = rows[tile_row<T>(i, g) * P + 16 * s + m];
#pragma unroll
        for (int j = 0; j < NG; ++j)
          acc[j][s] = mfma16x4(res[j][i], xc, acc[j][s]);
      }
    // the next rows overwrite the staged ones only after every lane has read
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // the waves' partial gradients meet in LDS; each wave adds a quarter of
  // them in wave order and stores it
  lptr<T> red = (lptr<T>)(T*)smem;
  lptr<double> sums = (lptr<double>)(double*)(smem + glm_tile_sums_at<T, NG>(S));
  constexpr int E = NG * S * 4;  // accumulators of a lane
  __syncthreads();               // every wave has read its staged rows
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    double v = sum[j];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (g == 0) sums[w * CT + 16 * j + m] = v;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        red[(w * E + (j * S + s) * 4 + i) * 64 + l] = acc[j][s][i];
  }
  __syncthreads();
  T* out = (T*)a.ws_grad + (size_t)slot * CT * a.width;
#pragma unroll
  for (int u = 0; u < E / kTileWaves; ++u) {
    const int x = w + kTileWaves * u;  // (j, s, i) = (u / S, u % S, w)
    const T v = ((red[x * 64 + l] + red[(E + x) * 64 + l]) +
                 red[(2 * E + x) * 64 + l]) + red[(3 * E + x) * 64 + l];
    out[(size_t)(16 * (u / S) + tile_row<T>(w, g)) * a.width + 16 * (u % S) +
        m] = v;
  }
  if (tid < CT)
    a.ws_sum[(size_t)slot * CT + tid] =
        ((sums[tid] + sums[CT + tid]) + sums[2 * CT + tid]) + sums[3 * CT + tid];
}

// Block b: a tile of 16 NG chains over one range of rows.  Blocks of one range
// are neighbours (one XCD, whose L2 then holds the range), or with a table
// those of one tile.  S is chosen from the problem's columns; SMAX bounds it,
// so that narrow launches take fewer registers.
template <typename T, int SMAX, int NG>
__global__ void __launch_bounds__(64 * kTileWaves, 2)
    glm_tile_grad(GlmTileArgs a, int want_sum) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int CT = 16 * NG;
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int ti = a.tiles ? b / a.n_split : b % a.n_tiles;
  const int split = a.tiles ? b % a.n_split : b / a.n_tiles;
  const GlmTile tile = glm_tile_of(a, ti, CT);
  if (split >= tile.n_split) return;
  const hipmc_problem& pb = a.problems[tile.prob];
  const int dx = pb.kind == HIPMC_TARGET_LINEAR ? pb.dim - 1 : pb.dim;
  const int ns = (dx + 15) >> 4;
  const int slot = tile.slot0 + split;
  const int row0 = split * tile.rows;
  const int row1 = row0 + tile.rows < pb.n_obs ? row0 + tile.rows : pb.n_obs;
  // a design the pass cannot read (rows not 16-byte aligned, a pitch below
  // the coefficients, an empty X), as in Target::glm, gives NaN
  if ((pb.x_pitch & 3) != 0 || pb.x_pitch < dx || dx < 1 || pb.n_obs < 1 ||
      ns > SMAX || 16 * ns > a.width) {
    for (int i = threadIdx.x; i < CT * a.width; i += blockDim.x)
      ((T*)a.ws_grad)[(size_t)slot * CT * a.width + i] = T(NAN);
    if ((int)threadIdx.x < CT)
      a.ws_sum[(size_t)slot * CT + threadIdx.x] = (double)NAN;
    return;
  }
  const bool ws = want_sum != 0;
#define HIPMC_TILE_CASE(S)                                                  \
  if constexpr (S <= SMAX) {                                                \
    if (ns == S) {                                                          \
      glm_tile_rows<T, S, NG>(pb, tile, a, row0, row1, ws, slot, smem_raw); \
      return;                                                               \
    }                                                                       \
  }
  HIPMC_TILE_CASE(1) HIPMC_TILE_CASE(2) HIPMC_TILE_CASE(3) HIPMC_TILE_CASE(4)
  HIPMC_TILE_CASE(5) HIPMC_TILE_CASE(6) HIPMC_TILE_CASE(7) HIPMC_TILE_CASE(8)
  HIPMC_TILE_CASE(9) HIPMC_TILE_CASE(10) HIPMC_TILE_CASE(11)
  HIPMC_TILE_CASE(12) HIPMC_TILE_CASE(13) HIPMC_TILE_CASE(14)
  HIPMC_TILE_CASE(15) HIPMC_TILE_CASE(16)
#undef HIPMC_TILE_CASE
}

// The row sums of one chain into tg, its ranges added in a fixed order.  `wpc`
// waves of the block share a chain (1, or 4 where there are many ranges), each
// taking consecutive ranges with up to U loads in flight; their sums meet in
// LDS (part 0's wave gets the total).  Every wave of the block calls it.
template <typename T, int K>
__device__ inline void load_row_sums(const GlmTileArgs& a, const GlmTile& tile,
                                     int local, int ct, int wpc, bool live,
                                     Target<T, K, kFamilyGlm, kRowSums>& tg) {
  constexpr int U = K * sizeof(T) <= 8 ? 16 : (K * sizeof(T) <= 16 ? 8 : 4);
  __shared__ T part_g[4][K * 64];
  __shared__ double part_s[4];
  const int lane = lane_id();
  const int wave = threadIdx.x >> 6;
  const int part = wpc > 1 ? wave : 0;
  const int n = live ? tile.n_split : 0;
  const int sp0 = n * part / wpc, sp1 = n * (part + 1) / wpc;
  const T* g0 = (const T*)a.ws_grad +
                ((size_t)tile.slot0 * ct + local) * a.width;
  const size_t step = (size_t)ct * a.width;
#pragma unroll
  for (int k = 0; k < K; ++k) tg.row_grad[k] = T(0);
  for (int sp = sp0; sp < sp1; sp += U) {
    T v[U][K];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int e = k * 64 + lane;
        v[u][k] = e < a.width && sp + u < sp1
                      ? g0[(size_t)(sp + u) * step + e] : T(0);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < K; ++k) tg.row_grad[k] += v[u][k];
  }
  double s = 0.0;
  for (int i = sp0 + lane; i < sp1; i += 64)
    s += a.ws_sum[((size_t)tile.slot0 + i) * ct + local];
  tg.row_sum = wave_sum(s);
  if (wpc > 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) part_g[wave][k * 64 + lane] = tg.row_grad[k];
    if (lane == 0) part_s[wave] = tg.row_sum;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int e = k * 64 + lane;
      tg.row_grad[k] = ((part_g[0][e] + part_g[1][e]) + part_g[2][e]) +
                       part_g[3][e];
    }
    tg.row_sum = ((part_s[0] + part_s[1]) + part_s[2]) + part_s[3];
  }
}

// Log density and gradient rows of every chain from the row sums.
template <typename T, int K>
__global__ void __launch_bounds__(256)
    glm_tile_finish(GlmTileArgs a, int ct, int wpc, T* out_tlp, T* out_grad) {
  const int wave = threadIdx.x >> 6;
  const int i = wpc > 1 ? blockIdx.x : blockIdx.x * 4 + wave;
  const int ti = i / ct, local = i - ti * ct;
  const bool has_tile = ti < a.n_tiles;
  const GlmTile tile = glm_tile_of(a, has_tile ? ti : 0, ct);
  const bool live = has_tile && local < tile.n_chains;
  const hipmc_problem& pb = a.problems[tile.prob];
  Target<T, K, kFamilyGlm, kRowSums> tg;
  tg.load(pb, nullptr);
  load_row_sums(a, tile, local, ct, wpc, live, tg);
  if (!live || (wpc > 1 && wave > 0)) return;
  const size_t c = tile.chain0 + local;
  T q[K], g[K];
  load_row(q, (const T*)a.x + c * a.stride, pb.dim);
  const double t = tg.eval(q, g);
  if (out_grad) store_row(out_grad + c * a.stride, g, pb.dim);
  if (lane_id() == 0 && out_tlp) out_tlp[c] = (T)t;
}

// The per-chain arithmetic of hmc_kernel between the all-chain gradients, for
// launches over one problem (no chain maps, no streams).  Positions and
// momenta of the trajectory live in ws_q (GlmTileArgs::x) and ws_p
// [n_chains, stride]; ws_ke0 [n_chains] holds the initial kinetic energy.
enum { kTileStart = 0, kTileMiddle = 1, kTileLast = 2 };

template <typename T, int K, bool CALIBRATED>
__global__ void __launch_bounds__(256)
    glm_tile_step(hipmc_run_args a, GlmTileArgs ta, int ct, int wpc, int mode,
                  int it, T* ws_p, double* ws_ke0) {
  const int lane = lane_id();
  const int wave = threadIdx.x >> 6;
  if (mode == kTileStart) wpc = 1;  // no sums to share
  const int ci = wpc > 1 ? blockIdx.x : blockIdx.x * 4 + wave;
  const bool live = ci < a.n_chains;
  if (mode == kTileStart && !live) return;
  const int c = live ? ci : a.n_chains - 1;
  const ChainId id = chain_of(a, c);
  const hipmc_problem& pb = a.problems[id.prob];
  const int dim = pb.dim;
  const size_t row = (size_t)c * a.dim_stride;
  T* qrow = (T*)ta.x + row;
  T* prow = ws_p + row;
  const T eps = load_step<T>(a, c);
  const T half = T(0.5) * eps;
  T m[K];
  double kconst;
  const bool pre = load_precision(a, id, dim, m, kconst);
  const Stream stream = stream_of(a, id.prob);
  const bool last_iter = it == stream.n_iters - 1;
  T q[K], p[K], g[K];
  if (mode == kTileStart) {
    const Seed sd = iter_seed(stream, it);
    draw_momentum(CALIBRATED ? split(sd, 0) : sd, id, dim, p);
    if (pre) precondition_momentum(m, p);
    if (last_iter && a.out_initial_momentum)
      store_row((T*)a.out_initial_momentum + row, p, dim);
    const double ke0 = half_kinetic(m, p);
    if (lane == 0) ws_ke0[c] = ke0;
    load_row(q, (const T*)a.state + row, dim);
    load_row(g, (const T*)a.grad + row, dim);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      p[k] = p[k] + half * g[k];
      q[k] = q[k] + eps * (m[k] * p[k]);
    }
    store_row(qrow, q, dim);
    store_row(prow, p, dim);
    return;
  }
  load_row(q, (const T*)qrow, dim);
  load_row(p, (const T*)prow, dim);
  Target<T, K, kFamilyGlm, kRowSums> tg;
  tg.load(pb, nullptr);
  const int ti = c / ct;
  load_row_sums(ta, glm_tile_of(ta, ti, ct), c - ti * ct, ct, wpc, live, tg);
  if (!live || (wpc > 1 && wave > 0)) return;
  double lpu;
  const double lpl = tg.eval_partial(q, g, lpu);
#pragma unroll
  for (int k = 0; k < K; ++k) p[k] = p[k] + eps * g[k];
  if (mode == kTileMiddle) {
#pragma unroll
    for (int k = 0; k < K; ++k) q[k] = q[k] + eps * (m[k] * p[k]);
    store_row(qrow, q, dim);
    store_row(prow, p, dim);
    return;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) p[k] = p[k] - half * g[k];
  const double t = wave_sum(lpl) + lpu;
  const double ke1 = half_kinetic(m, p);
  double corr = ws_ke0[c] - ke1;
  if (!__builtin_isfinite(corr)) corr = neg_inf();
  const size_t o = (size_t)(a.out_row0 + it) * a.n_chains + c;
  bool accept = true;
  double lar = 0.0;
  if (CALIBRATED) {
    const Seed acc = split(iter_seed(stream, it), 1);
    lar = (t - (double)((const T*)a.tlp)[c]) + corr;
    if (!__builtin_isfinite(lar)) lar = neg_inf();
    const U4 uw = philox(U4{0u, (uint32_t)id.local, id.key, kPurposeMHAccept},
                         acc.k0, acc.k1);
    accept = log((double)uniform_from<T>(uw.x, uw.y)) < lar;
    if (last_iter) {
      if (a.out_proposed_state)
        store_row((T*)a.out_proposed_state + row, q, dim);
      if (lane == 0) put<T>(a.out_proposed_tlp, c, (T)t);
    }
  }
  if (last_iter && a.out_final_momentum)
    store_row((T*)a.out_final_momentum + row, p, dim);
  if (accept) {
    store_row((T*)a.state + row, q, dim);
    store_row((T*)a.grad + row, g, dim);
  }
  if (lane == 0) {
    const T t1 = accept ? (T)t : ((const T*)a.tlp)[c];
    ((T*)a.tlp)[c] = t1;
    if (CALIBRATED) {
      put<T>(a.out_log_accept_ratio, o, (T)lar);
      if (a.out_is_accepted) a.out_is_accepted[o] = accept;
    }
    put<T>(a.out_energy, o, (T)corr);
    put<T>(a.out_target_log_prob, o, t1);
  }
  if (trace_row(stream, it) >= 0) {
    if (!accept) load_row(q, (const T*)a.state + row, dim);
    trace_store(stream, a, id, dim, it, q);
  }
}

}  // namespace hipmc
