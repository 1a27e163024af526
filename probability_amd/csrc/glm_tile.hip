// Launchers of the tiled GLM evaluation (glm_tile.h) for one state type;
// compiled once per type (HIPMC_INST_T).
#include "glm_tile.h"

#include "runtime.h"

#ifndef HIPMC_INST_T
#error "glm_tile.hip needs HIPMC_INST_T"
#endif

namespace hipmc {
namespace {

template <typename T, int SMAX, int NG>
int launch_grad(const GlmTileArgs& a, bool want_sum, hipStream_t s) {
  const size_t bytes = glm_tile_lds<T, NG>(a.width / 16);
  if (bytes > (size_t)kMaxLdsPerBlock) {
    const int rc = hip_check(
        hipFuncSetAttribute(
            reinterpret_cast<const void*>(&glm_tile_grad<T, SMAX, NG>),
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes),
        "hipFuncSetAttribute(max dynamic LDS)");
    if (rc != HIPMC_OK) return rc;
  }
  hipLaunchKernelGGL((glm_tile_grad<T, SMAX, NG>), dim3(a.n_tiles * a.n_split),
                     dim3(64 * kTileWaves), bytes, s, a, want_sum ? 1 : 0);
  return HIPMC_OK;
}

// The narrowest build that holds the launch's slabs.
template <typename T>
int grad(const GlmTileArgs& a, int ct, bool want_sum, hipStream_t s) {
  const int ns = a.width / 16;
  if (ct == 32) {
    if (ns <= 2) return launch_grad<T, 2, 2>(a, want_sum, s);
    if (ns <= 4) return launch_grad<T, 4, 2>(a, want_sum, s);
    if constexpr (sizeof(T) == 4) {
      if (ns <= 8) return launch_grad<T, 8, 2>(a, want_sum, s);
    }
  } else if (ct == 16) {
    if (ns <= 4) return launch_grad<T, 4, 1>(a, want_sum, s);
    if (ns <= 8) return launch_grad<T, 8, 1>(a, want_sum, s);
    if constexpr (sizeof(T) == 4) {
      if (ns <= 16) return launch_grad<T, 16, 1>(a, want_sum, s);
    }
  }
  return fail(HIPMC_E_UNSUPPORTED, "glm_tile: no kernel for this width");
}

// Waves that share a chain's row sums: with more than 16 ranges their loads
// are worth four waves' latency.
int waves_for(const GlmTileArgs& a) { return a.n_split > 16 ? 4 : 1; }

template <typename T, int K>
void finish(const GlmTileArgs& a, int ct, void* tlp, void* grad_out,
            hipStream_t s) {
  const int wpc = waves_for(a), chains = a.n_tiles * ct;
  hipLaunchKernelGGL((glm_tile_finish<T, K>),
                     dim3(wpc > 1 ? chains : (chains + 3) / 4), dim3(256), 0,
                     s, a, ct, wpc, (T*)tlp, (T*)grad_out);
}

template <typename T, int K, bool CAL>
void step(const hipmc_run_args& r, const GlmTileArgs& a, int ct, int mode,
          int it, void* ws_p, double* ws_ke0, hipStream_t s) {
  const int wpc = mode == kTileStart ? 1 : waves_for(a);
  hipLaunchKernelGGL((glm_tile_step<T, K, CAL>),
                     dim3(wpc > 1 ? r.n_chains : (r.n_chains + 3) / 4),
                     dim3(256), 0, s, r, a, ct, wpc, mode, it, (T*)ws_p,
                     ws_ke0);
}

}  // namespace

template <typename T>
int glm_tile_eval(const GlmTileArgs& a, int ct, int k, void* tlp,
                  void* grad_out, hipStream_t s) {
  const int rc = grad<T>(a, ct, true, s);
  if (rc != HIPMC_OK) return rc;
  switch (k) {
#define HIPMC_CASE(KK) \
  case KK: finish<T, KK>(a, ct, tlp, grad_out, s); break;
    HIPMC_CASE(1) HIPMC_CASE(2) HIPMC_CASE(3) HIPMC_CASE(4) HIPMC_CASE(5)
    HIPMC_CASE(8)
#undef HIPMC_CASE
    default: return fail(HIPMC_E_UNSUPPORTED, "glm_tile: no kernel");
  }
  return hip_check(hipGetLastError(), "glm_tile evaluation launch");
}

template <typename T>
int glm_tile_hmc(const hipmc_run_args& r, const GlmTileArgs& a, int ct, int k,
                 bool calibrated, void* ws_p, double* ws_ke0, hipStream_t s) {
  auto go = [&](int mode, int it) {
    switch (k) {
#define HIPMC_CASE(KK)                                               \
  case KK:                                                           \
    if (calibrated)                                                  \
      step<T, KK, true>(r, a, ct, mode, it, ws_p, ws_ke0, s);        \
    else                                                             \
      step<T, KK, false>(r, a, ct, mode, it, ws_p, ws_ke0, s);       \
    return HIPMC_OK;
      HIPMC_CASE(1) HIPMC_CASE(2) HIPMC_CASE(3) HIPMC_CASE(4) HIPMC_CASE(5)
      HIPMC_CASE(8)
#undef HIPMC_CASE
    }
    return fail(HIPMC_E_UNSUPPORTED, "glm_tile: no kernel");
  };
  for (int it = 0; it < r.n_iters; ++it) {
    int rc = go(kTileStart, it);
    if (rc != HIPMC_OK) return rc;
    for (int st = 0; st < r.num_leapfrog_steps; ++st) {
      const bool last = st + 1 == r.num_leapfrog_steps;
      // the log density is needed at the trajectory's end only
      rc = grad<T>(a, ct, last, s);
      if (rc != HIPMC_OK) return rc;
      go(last ? kTileLast : kTileMiddle, it);
    }
  }
  return hip_check(hipGetLastError(), "glm_tile trajectory launch");
}

template int glm_tile_eval<HIPMC_INST_T>(const GlmTileArgs&, int, int, void*,
                                         void*, hipStream_t);
template int glm_tile_hmc<HIPMC_INST_T>(const hipmc_run_args&,
                                        const GlmTileArgs&, int, int, bool,
                                        void*, double*, hipStream_t);

}  // namespace hipmc
