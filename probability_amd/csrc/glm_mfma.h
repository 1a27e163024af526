// Large-batch HMC for Bayesian logistic regression with the design matrix
// stored in BF16 and the all-chain contraction on MFMA (gfx950
// v_mfma_f32_32x32x16_bf16).
//
// One leapfrog gradient for C chains (`mcmc/hmc.py` target gradient through
// `mcmc/internal/util.py:246-308`, Bernoulli logits `bernoulli.py:119-135`):
//   S = X B^T            [N x C]   (B = chain positions, split B = Bhi + Blo)
//   R = y - sigmoid(S)   [N x C]   (split R = Rhi + Rlo)
//   G = R^T X            [C x D]   (+ prior gradient in the update kernel)
// glm_grad_mfma fuses both GEMMs per tile of 32 rows: the tile of X (and of
// X^T) is staged in LDS once and used for both products, S and R never
// leave registers/LDS (no [N x C] array in HBM), and each workgroup writes
// one partial G for its row range (split-N), reduced in fixed order by the
// per-chain update kernel.  FP32 accumulation throughout; the BF16 hi/lo
// split of B and R keeps ~16 mantissa bits of both operands that are not
// data.
#pragma once

#include <type_traits>

#include "../../include/hipmc.h"
#include "common.h"

namespace hipmc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kMD = 256;       // state dimension of this path
constexpr int kMRows = 32;     // rows per LDS tile
constexpr int kMChains = 64;   // chain granularity of the path (32 per wave)
constexpr int kRPitch = kMRows + 8;    // bf16 per R row (one chain) in LDS

// D += A B with A 32 x 16, B 16 x 32: lane l holds row l % 32 of A and column
// l % 32 of B at k = 8 (l / 32) + [0, 8); register r of D is row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
// The unit adds its products to the accumulator in groups of 8 in the order
// of k, so two of these in a row give bit for bit what one
// v_mfma_f32_16x16x32_bf16 of the same 32 columns gives.
__device__ inline f32x16 mfma32(const bf16x8& a, const bf16x8& b,
                                const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Where element e of chain c stands in Bhi and Blo: in the order in which the
// gradient's waves read their fragments, 32 chains by 16 elements per KiB.
// (Read from rows, a load of 16 bytes per lane touched 32 cache lines, and a
// launch with one tile per workgroup took 1 us longer.)
__device__ inline size_t coef_index(int c, int e) {
  return (size_t)(c >> 5) * 32 * kMD +
         (((e >> 4) * 64 + ((e >> 3) & 1) * 32 + (c & 31)) * 8 + (e & 7));
}

// two floats rounded to BF16, the first in the low half
__device__ inline uint32_t pack_bf16(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Direct global -> LDS loads (global_load_lds): the wave's 64 lanes each
// read 16 (or 4) bytes from their own address and the bytes land at the
// wave-uniform LDS base + 16 (4) * lane.  Issued from inline asm so that the
// compiler's wait-count pass does not make every later LDS read wait for
// them; the kernel waits for its own tile loads (vmcnt) before the barrier
// that publishes a tile.  m0 is a reserved register whose clobber the
// compiler does not track (hipcc warns): each asm statement sets m0 and
// issues the load that reads it, and nothing else in glm_grad_mfma uses m0
// (no LDS-DMA builtins, no dynamically indexed register arrays), which the
// gfx950 assembly of the kernel confirms (its only m0 writes are these).
typedef __attribute__((address_space(3))) char lds_byte;
typedef const __attribute__((address_space(3))) bf16x8 lds_bf16x8;
__device__ inline uint32_t lds_addr(void* p) {
  return (uint32_t)(uintptr_t)(lds_byte*)p;
}
__device__ inline void lds_dma16(const void* g, void* lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(g), "s"(lds_addr(lds_base)) : "memory", "m0");
}
// the same from a wave-uniform address plus 32-bit lane offsets
__device__ inline void lds_dma16(const void* g, uint32_t off, void* lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(g), "s"(lds_addr(lds_base))
               : "memory", "m0");
}
__device__ inline void lds_dma4(const void* g, uint32_t off, void* lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1"
               :: "v"(off), "s"(g), "s"(lds_addr(lds_base))
               : "memory", "m0");
}

// Chunk swizzle of X^T row d: 16 consecutive d of one chunk column land in
// 16 distinct 16-byte bank groups, and any 8 consecutive aligned d in 8.
__device__ inline int xt_swz(int d) { return ((d >> 1) ^ (d >> 2)) & 3; }

// What a lane loads of each tile.  X tile: 16-byte chunk (row, c) at chunk
// row * 32 + (c ^ (row & 15)); X^T tile: chunk (d, c) at d * 4 + (c ^
// xt_swz(d)).  The WAVES waves of the workgroup share a tile's 1024 chunk
// loads and its 32 labels.  The lane's part of an address is the same for
// every tile and is kept (it was some 130 integer instructions a tile).
template <int WAVES>
struct TileLoads {
  static constexpr int U = 16 / WAVES;       // 1 KiB chunk rows per wave
  static constexpr int YL = kMRows / WAVES;  // labels per wave
  int w, l;
  uint32_t xoff[U];  // within a tile of X
  uint64_t xt0;      // this lane's first chunk of tile 0 of X^T
  size_t xt_step;    // bytes of 16 rows of X^T
  __device__ TileLoads(const __bf16* Xt, int n_obs, int wave, int lane)
      : w(__builtin_amdgcn_readfirstlane(wave)), l(lane) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = (w * U + u) * 64 + l;
      const int row = q >> 5, c = (q & 31) ^ (row & 15);
      xoff[u] = (uint32_t)(row * kMD + c * 8) * 2;
    }
    // rows d = 16 (w U + u) + l / 4: the swizzle repeats every 16
    const int d = w * U * 16 + (l >> 2), c = (l & 3) ^ xt_swz(l >> 2);
    xt0 = (uint64_t)(Xt + (size_t)d * n_obs + c * 8);
    xt_step = (size_t)n_obs * 32;
  }
  __device__ void x(const __bf16* X, int n0, __bf16* xs) const {
    const __bf16* g = X + (size_t)n0 * kMD;
#pragma unroll
    for (int u = 0; u < U; ++u)
      lds_dma16(g, xoff[u], (char*)xs + (w * U + u) * 1024);
  }
  __device__ void xt(int n0, __bf16* xts) const {
    const uint64_t g = xt0 + (size_t)n0 * 2;
#pragma unroll
    for (int u = 0; u < U; ++u)
      lds_dma16((const void*)(g + u * xt_step),
                (char*)xts + (w * U + u) * 1024);
  }
  __device__ void labels(const float* y, int n0, float* ys) const {
    if (l < YL) lds_dma4(y + n0 + w * YL, l * 4, ys + w * YL);
  }
};

// Partial gradient (and with LL the partial Bernoulli log-likelihood, which a
// trajectory's last gradient needs) of the chains [32*WAVES*blockIdx.x,
// +32*WAVES) over rows [blockIdx.y*rows_per_split, +rows), 32 chains per wave,
// one wave per SIMD (its coefficients and gradients take 256 registers).
//
// What bounds it: the matrix unit at the clock the card holds under it.
// 32x32x16 MFMAs run at 2.23 PFLOP/s here by themselves, 16x16x32 ones (16
// chains per wave, the layout before) at no more than 1.66, and beside those
// every VALU instruction adds its whole issue time, while a 32x32x16 hides
// about four.  So the kernel runs ahead: a step takes the logits of tile t + 2,
// the residuals of tile t + 1 and the gradient of tile t, which do not depend
// on each other, two residuals beside every eight products.  65536 x 256, 4096
// chains (both products with hi and lo parts, 550 GFLOP): 515 -> 470 us, 1.17
// PFLOP/s, where a large BF16 matrix product reaches 1.13; the matrix unit was
// busy for 47% of the cycles and is for 60%, at a clock that falls from 2.0 to
// 1.9 GHz, so that other orders of the same instructions measured the same and
// fewer instructions less.  An HMC transition, L = 20: 10.59 -> 9.66 ms; of
// 8192 rows and 64 chains 421 -> 412 us.  The sums are the same bit for bit.
//
// Tiles of 32 rows of X and X^T go straight from memory to LDS (no
// registers).  X is staged two tiles ahead of X^T, each in two buffers, and one
// barrier a step serves both as "the loads of the last step have landed" and
// "every wave has left the buffers that this step's loads overwrite".
// LDS layouts (16-byte chunks, XOR-swizzled so that the MFMA fragment reads of
// eight consecutive rows hit distinct banks): X tile chunk (row, c) at row * 32
// + (c ^ (row & 15)), X^T tile chunk (d, c) at d * 4 + (c ^ xt_swz(d)).  Each
// lane writes four consecutive residual rows as one 8-byte store (R pitch 40
// bf16 keeps those stores and the 16-byte fragment reads free of conflicts).
template <int WAVES, bool LL>
__global__ void __launch_bounds__(64 * WAVES, 1)
    glm_grad_mfma(const __bf16* __restrict__ X, const __bf16* __restrict__ Xt,
                  const float* __restrict__ y, int n_obs,
                  const __bf16* __restrict__ Bhi,
                  const __bf16* __restrict__ Blo, int n_chains,
                  int rows_per_split, float* __restrict__ out_g,
                  float* __restrict__ out_ll) {
  constexpr int kTile = kMRows * kMD;
  constexpr int KB = kMD / 32;     // 32-column blocks
  constexpr int NT = kMD / 32;     // 32-coefficient gradient tiles
  static_assert(KB == NT, "one block of each in a scheduling region");
  constexpr int CH = 32 * WAVES;   // chains of the workgroup
  __shared__ __align__(1024) __bf16 xs[2 * kTile];
  __shared__ __align__(1024) __bf16 xts[2 * kTile];
  __shared__ __align__(16) __bf16 rs[2 * CH * kRPitch];
  __shared__ __align__(16) float ys[2 * kMRows];
  const int tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, m = l & 31, h = l >> 5;
  const int c0 = blockIdx.x * CH + 32 * w;
  const int r0 = blockIdx.y * rows_per_split;
  const int r1 = min(n_obs, r0 + rows_per_split);
  const int tiles = (r1 - r0) / kMRows;
  const TileLoads<WAVES> load(Xt, n_obs, w, l);
  if (tiles > 0) {
    load.x(X, r0, xs);
    load.labels(y, r0, ys);
    load.xt(r0, xts);
    if (tiles > 1) {
      load.x(X, r0 + kMRows, xs + kTile);
      load.labels(y, r0 + kMRows, ys + kMRows);
    }
  }
  // coefficients of chain m, columns 16 k + 8 h + [0, 8): 1 KiB per load
  bf16x8 bh[2 * KB], bl[2 * KB];
#pragma unroll
  for (int k = 0; k < 2 * KB; ++k) {
    const size_t off = coef_index(c0 + m, 16 * k + 8 * h);
    bh[k] = *(const bf16x8*)(Bhi + off);
    bl[k] = *(const bf16x8*)(Blo + off);
  }
  // keep the fragments in registers (not re-read from memory per tile,
  // whose waits would also wait for the tile loads in flight)
#pragma unroll
  for (int k = 0; k < 2 * KB; ++k) asm volatile("" : "+v"(bh[k]), "+v"(bl[k]));
  f32x16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nt][r] = 0.f;
  // log-likelihood of the lane's rows, kept as the sums of rows 4 h + [0, 4)
  // (mod 16) and 8 + 4 h + [0, 4) (mod 16)
  float lls[2] = {0.f, 0.f};
  __bf16* rh_w = rs + (32 * w + m) * kRPitch;
  __bf16* rl_w = rh_w + CH * kRPitch;

  // row m of a tile, 16-byte chunk 2 k + h, which sits at (2 k + h) ^ (m % 16)
  // = 16 (k / 8) + (2 (k % 8) + h) ^ (m % 16): eight lane addresses, the rest
  // are constants
  int xo[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) xo[b] = (m * 32 + ((2 * b + h) ^ (m & 15))) * 8;
  auto x_frag = [&](const __bf16* x, int k) {
    return *(const bf16x8*)&x[xo[k & 7] + 16 * (k >> 3) * 8];
  };
  uint32_t xo_t[2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
    xo_t[k] = (m * 4 + ((2 * k + h) ^ xt_swz(m))) * 16;
  // residual (and log-likelihood) of one logit
  auto residual = [&](float sv, float yv, float& ll) {
    const float e = __expf(-fabsf(sv));
    const float inv = recip_1p(e);
    const float sig = sv >= 0.f ? inv : e * inv;
    if (LL) {
      const float sp_abs = log1p_unit(e);
      const float sp_pos = sp_abs + fmaxf(sv, 0.f);
      const float sp_neg = sp_abs + fmaxf(-sv, 0.f);
      const float w0 = 1.f - yv;
      ll += (w0 == 0.f ? 0.f : -sp_pos * w0) + (yv == 0.f ? 0.f : -sp_neg * yv);
    }
    return yv - sig;
  };
  // residuals of the tile behind the logits, and the fragments the gradient
  // reads: chain m, rows 16 k + 8 h + [0, 8)
  bf16x8 ah0, ah1, al0, al1;
  f32x16 s;
  // one step: S logits of the tile in xn (into s), R residuals of the tile
  // whose logits s holds, G gradient of the tile in xt whose residuals are in
  // ah and al.  The three are independent; the scheduling barriers keep a
  // block's fragment reads one block ahead of its products and two residuals
  // beside each block of eight.
  auto step = [&](auto do_s, auto do_r, auto do_g, const __bf16* xn,
                  const __bf16* xt, const float* yt) {
    constexpr bool S = decltype(do_s)::value, R = decltype(do_r)::value,
                   G = decltype(do_g)::value;
    const uint32_t xt_base = G ? lds_addr((void*)xt) : 0;
    f32x16 n;
#pragma unroll
    for (int r = 0; r < 16; ++r) n[r] = 0.f;
    // chunks 2 k + h of X^T row 32 nt + m: two lane addresses (opaque, or the
    // compiler keeps and adds sixteen)
    uint32_t xa[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      xa[k] = xt_base + xo_t[k];
      asm volatile("" : "+v"(xa[k]));
    }
    auto xt_frag = [&](int nt, int k) {
      return *(lds_bf16x8*)(uintptr_t)(xa[k] + 2048 * nt);
    };
    uint32_t hv = 0, lv = 0;
    f32x4 yv;
    bf16x8 a0, a1, t0, t1;
    if (S) {
      a0 = x_frag(xn, 0);
      a1 = x_frag(xn, 1);
    }
    if (G) {
      t0 = xt_frag(0, 0);
      t1 = xt_frag(0, 1);
    }
    if (R) yv = *(const f32x4*)&yt[4 * h];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      bf16x8 b0, b1, u0, u1;
      f32x4 yn;
      if (S && kb + 1 < KB) {
        b0 = x_frag(xn, 2 * kb + 2);
        b1 = x_frag(xn, 2 * kb + 3);
      }
      if (G && kb + 1 < NT) {
        u0 = xt_frag(kb + 1, 0);
        u1 = xt_frag(kb + 1, 1);
      }
      const int q = kb >> 1;  // rows 8 q + 4 h + [0, 4)
      if (R && (kb & 1) && kb + 1 < KB)
        yn = *(const f32x4*)&yt[8 * q + 8 + 4 * h];
      if (S) n = mfma32(a0, bh[2 * kb], n);
      if (G) acc[kb] = mfma32(ah0, t0, acc[kb]);
      if (S) n = mfma32(a1, bh[2 * kb + 1], n);
      if (G) acc[kb] = mfma32(ah1, t1, acc[kb]);
      if (S) n = mfma32(a0, bl[2 * kb], n);
      if (G) acc[kb] = mfma32(al0, t0, acc[kb]);
      if (S) n = mfma32(a1, bl[2 * kb + 1], n);
      if (G) acc[kb] = mfma32(al1, t1, acc[kb]);
      if (R) {
        const int i = 2 * (kb & 1);
        const float ra = residual(s[4 * q + i], yv[i], lls[q & 1]);
        const float rb = residual(s[4 * q + i + 1], yv[i + 1], lls[q & 1]);
        const uint32_t hi = pack_bf16(ra, rb);
        const uint32_t lo = pack_bf16(ra - __uint_as_float(hi << 16),
                                      rb - __uint_as_float(hi & 0xffff0000u));
        if (kb & 1) {
          *(uint2*)&rh_w[8 * q + 4 * h] = make_uint2(hv, hi);
          *(uint2*)&rl_w[8 * q + 4 * h] = make_uint2(lv, lo);
        }
        hv = hi;
        lv = lo;
      }
      if (S) {
        a0 = b0;
        a1 = b1;
      }
      if (G) {
        t0 = u0;
        t1 = u1;
      }
      if (R && (kb & 1)) yv = yn;
      __builtin_amdgcn_sched_barrier(0);
    }
    if (S) s = n;
    if (R) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      ah0 = *(const bf16x8*)&rh_w[8 * h];
      ah1 = *(const bf16x8*)&rh_w[16 + 8 * h];
      al0 = *(const bf16x8*)&rl_w[8 * h];
      al1 = *(const bf16x8*)&rl_w[16 + 8 * h];
    }
  };
  using Yes = std::true_type;
  using No = std::false_type;
  auto landed = [&] {
    __builtin_amdgcn_s_waitcnt(0xF70);  // this wave's tile loads (vmcnt)
    __syncthreads();
  };
  // Step t: logits of tile t + 2, residuals of t + 1, gradient of t.  Buffer
  // j & 1 holds tile j of X, X^T and y; the loads a step issues replace what
  // the step before it read: X of t + 3, X^T of t + 1, y of t + 2.
  if (tiles > 0) {
    landed();
    step(Yes{}, No{}, No{}, xs, nullptr, nullptr);
    if (tiles > 1) {
      landed();
      if (tiles > 2) load.x(X, r0 + 2 * kMRows, xs);
      step(Yes{}, Yes{}, No{}, xs + kTile, nullptr, ys);
    } else {
      step(No{}, Yes{}, No{}, nullptr, nullptr, ys);
    }
  }
  for (int t = 0; t + 2 < tiles; ++t) {
    landed();
    const int n0 = r0 + t * kMRows;
    const int b = t & 1, o = b ^ 1;
    if (t + 3 < tiles) load.x(X, n0 + 3 * kMRows, xs + o * kTile);
    load.xt(n0 + kMRows, xts + o * kTile);
    load.labels(y, n0 + 2 * kMRows, ys + b * kMRows);
    step(Yes{}, Yes{}, Yes{}, xs + b * kTile, xts + b * kTile,
         ys + o * kMRows);
  }
  if (tiles > 1) {
    landed();
    const int b = tiles & 1, o = b ^ 1;
    load.xt(r0 + (tiles - 1) * kMRows, xts + o * kTile);
    step(No{}, Yes{}, Yes{}, nullptr, xts + b * kTile, ys + o * kMRows);
  }
  if (tiles > 0) {
    if (tiles > 1) landed();
    step(No{}, No{}, Yes{}, nullptr, xts + ((tiles - 1) & 1) * kTile, nullptr);
  }
  float* og = out_g + ((size_t)blockIdx.y * n_chains + c0) * kMD;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      og[(size_t)(8 * (r >> 2) + 4 * h + (r & 3)) * kMD + 32 * nt + m] =
          acc[nt][r];
  if (LL) {
    const float p = lls[0] + __shfl_xor(lls[0], 32);
    const float q = lls[1] + __shfl_xor(lls[1], 32);
    if (h == 0) out_ll[(size_t)blockIdx.y * n_chains + c0 + m] = p + q;
  }
}
// ---------------------------------------------------------------- per chain
// One block of 256 threads per chain, thread e holds state element e.
__device__ inline void split_bf16(float v, __bf16& hi, __bf16& lo) {
  hi = (__bf16)v;
  lo = (__bf16)(v - (float)hi);
}

__device__ inline float mfma_step_size(const hipmc_glm_hmc_args& a, int c) {
  return a.step_size[a.per_chain_step ? c : 0];
}

__device__ inline Seed mfma_iter_seed(const hipmc_glm_hmc_args& a, int it) {
  Seed base{a.seed[0], a.seed[1]};
  return a.fold_seed ? fold_in(base, (uint64_t)(a.iter0 + it)) : base;
}

// Writes Bhi/Blo of the current state (bootstrap gradient input).
__global__ void mfma_prepare(hipmc_glm_hmc_args a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)a.n_chains * kMD) return;
  __bf16 hi, lo;
  split_bf16(a.state[i], hi, lo);
  const size_t o = coef_index((int)(i / kMD), (int)(i % kMD));
  ((__bf16*)a.ws_b)[o] = hi;
  ((__bf16*)a.ws_b)[(size_t)a.n_chains * kMD + o] = lo;
}

// Element e of chain c: the split-N partial gradients added in split order,
// plus the prior.  The adds form a serial chain, the loads do not: kU of them
// are in flight at a time (a few chains take up to N / 32 splits, whose
// partial sums come from the other XCDs through memory).
__device__ inline float reduce_grad(const hipmc_glm_hmc_args& a, int c, int e,
                                    float q, float inv_ps2) {
  constexpr int kU = 32;
  const float* g = a.ws_g + (size_t)c * kMD + e;
  const size_t stride = (size_t)a.n_chains * kMD;
  const int n = a.n_split;
  float s = 0.f;
  int sp = 0;
  for (; sp + kU <= n; sp += kU) {
    float v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) v[u] = g[(size_t)(sp + u) * stride];
#pragma unroll
    for (int u = 0; u < kU; ++u) s += v[u];
  }
  for (; sp + 8 <= n; sp += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = g[(size_t)(sp + u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; sp < n; ++sp) s += g[(size_t)sp * stride];
  return s - q * inv_ps2;
}

// The splits' partial log-likelihoods added in split order (one wave; 64
// splits are loaded at once, one per lane).
__device__ inline double reduce_ll(const hipmc_glm_hmc_args& a, int c,
                                   int lane) {
  double s = 0.0;
  for (int sp = 0; sp < a.n_split; sp += 64) {
    const int m = a.n_split - sp < 64 ? a.n_split - sp : 64;
    const float v =
        lane < m ? a.ws_ll[(size_t)(sp + lane) * a.n_chains + c] : 0.f;
    for (int l = 0; l < m; ++l) s += (double)readlane_f(v, l);
  }
  return s;
}

// Wave 0's share of a block sum: elements lane, 64 + lane, 128 + lane and
// 192 + lane of v in that order, then over the lanes.
__device__ inline double element_sum(const double* v, int lane) {
  return wave_sum(((v[lane] + v[64 + lane]) + v[128 + lane]) + v[192 + lane]);
}

// mode 0: start of iteration `it` (momentum draw, first half kick, first
// drift); mode 1: after a gradient of a middle leapfrog step (kick, drift);
// mode 2: after the last gradient (kick, un-kick, MH accept); mode 3:
// bootstrap (tlp and grad of the state).
// Bound by reading the partial gradients [n_split, chains, 256]: few chains
// come with many splits, so a thread holds one element (four waves a chain)
// with up to 32 loads in flight.  Against one wave a chain with dependent
// loads, us per launch: 64 chains x 256 splits 228 -> 7.1 (17 MB, 2.4 TB/s);
// 4096 chains x 8 splits 15.1 -> 12.9.  The sums' order is the same.
__global__ void __launch_bounds__(kMD) mfma_chain_step(hipmc_glm_hmc_args a,
                                                       int mode, int it) {
  __shared__ double red[2][kMD];
  __shared__ double sums[2];
  const int e = threadIdx.x;
  const int lane = e & 63;
  const bool first = e < 64;  // wave 0 does the chain's scalar work
  const int c = blockIdx.x;
  const float ps = (float)a.prior_scale;
  const float inv_ps = 1.f / ps;
  const float inv_ps2 = inv_ps * inv_ps;
  const size_t row = (size_t)c * kMD;
  float* q = a.ws_q + row;
  float* p = a.ws_p + row;
  __bf16* bh = (__bf16*)a.ws_b + coef_index(c, e);
  __bf16* bl = bh + (size_t)a.n_chains * kMD;
  if (mode == 3) {
    const float qv = a.state[row + e];
    a.grad[row + e] = reduce_grad(a, c, e, qv, inv_ps2);
    const float z = qv * inv_ps;
    red[0][e] = (double)(-0.5f * z * z);
    __syncthreads();
    if (first) {
      const double lp = element_sum(red[0], lane);
      const double ll = reduce_ll(a, c, lane);
      if (lane == 0)
        a.tlp[c] = (float)(lp + ll +
                           kMD * (-0.9189385332046727 - log((double)ps)));
    }
    return;
  }
  const float eps = mfma_step_size(a, c);
  const float half = 0.5f * eps;
  const Seed sd = mfma_iter_seed(a, it);
  if (mode == 0) {
    const Seed prop = split(sd, 0);
    const U4 w = philox(U4{(uint32_t)(e >> 2), (uint32_t)c, a.key,
                           kPurposeMomentum},
                        prop.k0, prop.k1);
    const bool hi_pair = (e & 2) != 0;
    double n0, n1;
    box_muller(hi_pair ? w.z : w.x, hi_pair ? w.w : w.y, n0, n1);
    const float pv0 = (float)((e & 1) ? n1 : n0);
    const float pv = pv0 + half * a.grad[row + e];
    const float qv = a.state[row + e] + eps * pv;
    p[e] = pv;
    q[e] = qv;
    __bf16 hi, lo;
    split_bf16(qv, hi, lo);
    *bh = hi;
    *bl = lo;
    red[0][e] = (double)pv0 * (double)pv0;
    __syncthreads();
    if (first) {
      const double ke = element_sum(red[0], lane);
      if (lane == 0) a.ws_ke0[c] = 0.5 * ke;
    }
    return;
  }
  const float qv = q[e];
  const float gv = reduce_grad(a, c, e, qv, inv_ps2);
  if (mode == 1) {
    const float pv = p[e] + eps * gv;
    const float qn = qv + eps * pv;
    p[e] = pv;
    q[e] = qn;
    __bf16 hi, lo;
    split_bf16(qn, hi, lo);
    *bh = hi;
    *bl = lo;
    return;
  }
  // mode 2: last kick, un-kick, kinetic energy, log-prob, MH accept
  float pv = p[e] + eps * gv;
  pv = pv - half * gv;
  const float z = qv * inv_ps;
  red[0][e] = (double)pv * (double)pv;
  red[1][e] = (double)(-0.5f * z * z);
  __syncthreads();
  if (first) {
    const double ke = element_sum(red[0], lane);
    const double lp = element_sum(red[1], lane);
    const double ll = reduce_ll(a, c, lane);
    const double t1 = lp + ll +
                      kMD * (-0.9189385332046727 - log((double)ps));
    const double t0 = (double)a.tlp[c];
    double corr = a.ws_ke0[c] - 0.5 * ke;
    if (!__builtin_isfinite(corr)) corr = -__builtin_inf();
    double lar = (t1 - t0) + corr;
    if (!__builtin_isfinite(lar)) lar = -__builtin_inf();
    if (lane == 0) {
      sums[0] = t1;
      sums[1] = lar;
    }
  }
  __syncthreads();
  const double t1 = sums[0], lar = sums[1];
  const Seed acc = split(sd, 1);
  const U4 uw = philox(U4{0u, (uint32_t)c, a.key, kPurposeMHAccept}, acc.k0,
                       acc.k1);
  const bool accept = log((double)uniform_from<float>(uw.x, uw.y)) < lar;
  if (accept) {
    a.state[row + e] = qv;
    a.grad[row + e] = gv;
  }
  if (e == 0) {
    if (accept) a.tlp[c] = (float)t1;
    const size_t o = (size_t)it * a.n_chains + c;
    if (a.out_log_accept_ratio) a.out_log_accept_ratio[o] = (float)lar;
    if (a.out_is_accepted) a.out_is_accepted[o] = accept;
  }
  if (a.trace_state) {
    const int64_t gi = a.iter0 + it - a.trace_start;
    const int every = a.trace_every > 0 ? a.trace_every : 1;
    if (gi >= 0 && gi % every == 0 && gi / every < a.n_trace) {
      float* tr = a.trace_state + ((size_t)(gi / every) * a.n_chains + c) * kMD;
      tr[e] = accept ? qv : a.state[row + e];
    }
  }
}

}  // namespace hipmc
