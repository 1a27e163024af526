// Internal declarations shared by the library's translation units: the
// thread-local error message, HIP error checks, and the launchers of the
// sampling kernels.  Each (dtype, target family) pair of the sampling
// kernels is compiled in its own object (inst.hip), so the launchers are
// declared here and defined by explicit instantiation there.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <string>

#include "../../include/hipmc.h"

namespace hipmc {

// Sets the thread-local message returned by hipmc_last_error; returns code.
int fail(int code, const std::string& msg);
// HIPMC_OK, or HIPMC_E_HIP with the runtime's message.
int hip_check(hipError_t e, const char* what);

inline hipStream_t as_stream(uint64_t s) {
  return reinterpret_cast<hipStream_t>(s);
}

constexpr int kMaxLdsPerBlock = 64 * 1024;
// gfx950 gives one workgroup up to 160 KiB of LDS; a launch that asks for
// more than 64 KiB raises the kernel's dynamic-LDS limit first.
constexpr int kMaxLdsSharedChain = 160 * 1024;

// Register slots per lane (state elements / 64) built for a target family:
// up to 8 for GLMs, whose chains keep a second copy of their vectors parked
// in LDS, and up to 17 (1088 elements) for the others.
constexpr int max_slots(int fam) { return fam == 1 ? 8 : 17; }
// Smallest compiled slot count K of family fam with K*64 >= max_dim, or -1.
int pick_k(int max_dim, int fam);
// The largest state dimension built for family fam.
int max_state_dim(int fam);

// Sampling-kernel launchers of one (dtype T, family FAM) pair; k is the
// register slot count from pick_k.
template <typename T, int FAM>
int launch_nuts_k(int k, const hipmc_run_args& a, int32_t* queue,
                  const int32_t* order, hipStream_t s);
template <typename T, int FAM>
int launch_hmc_k(int k, bool calibrated, const hipmc_run_args& a,
                 hipStream_t s);
template <typename T, int FAM>
int launch_eval_k(int k, const hipmc_problem* p, const int32_t* cp, int n,
                  int stride, const void* x, void* tlp, void* grad,
                  hipStream_t s);

// The tiled GLM evaluation (glm_tile.h): blocks of kTileWaves waves.
constexpr int kTileWaves = 4;
// Rows of a block's pass over its range: 16 per wave.
constexpr int kTileRows = 16 * kTileWaves;

// One tile of chains of a batch (device table, [n_tiles]); a launch over one
// problem has none and works its tiles out.
struct GlmTile {
  int32_t prob, chain0, n_chains, n_split, slot0, rows, pad0_, pad1_;
};
static_assert(sizeof(GlmTile) == 32, "GlmTile layout");

struct GlmTileArgs {
  const hipmc_problem* problems;
  const GlmTile* tiles;  // NULL: tiles of problem 0
  int n_tiles, n_split;  // n_split: of every tile (NULL table) or the most
  int rows;              // rows per split (NULL table)
  int n_chains, stride;  // positions x [n_chains, stride]
  int width;             // workspace row of a chain (16 * slabs)
  const void* x;
  void* ws_grad;    // T [slots, tile chains, width]
  double* ws_sum;   // [slots, tile chains]
};

// Log density and gradient of every chain of the tiles; trajectories of a
// run over one problem (glm_tile.hip).  ct: chains per tile (16 or 32); k:
// register slots of the per-chain kernels.
template <typename T>
int glm_tile_eval(const GlmTileArgs& a, int ct, int k, void* tlp,
                  void* grad_out, hipStream_t s);
template <typename T>
int glm_tile_hmc(const hipmc_run_args& r, const GlmTileArgs& a, int ct, int k,
                 bool calibrated, void* ws_p, double* ws_ke0, hipStream_t s);

// The BF16 MFMA logistic-regression HMC path (mfma.hip), with caller
// workspaces or with the library's static scratch.
int launch_glm_hmc(const hipmc_glm_hmc_args* a, hipStream_t s);
int launch_glm_hmc_noalloc(const hipmc_glm_hmc_args* a, hipStream_t s);

}  // namespace hipmc
