"""When a regression's chains take the tiled evaluation (csrc/glm_tile.h: the
logits and gradients of many chains as matrix products over row ranges), and
its workspaces.

The other path is the sampling kernels' own: one chain per wave (up to four
waves per chain in HMC) passing over X by itself, one launch for a whole
trajectory.  The tiled one pays two launches per gradient, about 9 to 16 us
however small the problem, and 7 us more of host time per evaluation.  Where
the lines lie, us per call (evaluations, one after the other) or per leapfrog
step (four transitions of ten steps in a launch), one chain per wave / tiled,
MI355X:

  evaluation  float32  logistic   512 x 30,  256 chains   12.2 / 17.0
                                  800 x 30,  1 chain      16.6 / 16.9
                                  1200 x 8,  1 chain      18.5 / 16.8
                       linear     512 x 16,  4096 chains  26.4 / 17.1
                                  800 x 128, 64 chains    20.5 / 18.6
              float64  logistic   128 x 100, 64 chains    14.5 / 17.2
                                  512 x 64,  64 chains    24.2 / 18.0
                       linear     1300 x 30, 1 chain      19.2 / 21.1
                                  512 x 100, 64 chains    23.7 / 17.1
  trajectory  float32  logistic   512 x 8,   2000 chains  10.5 / 11.5
                                  2048 x 8,  256 chains    9.2 / 10.6
                                  3000 x 30, 256 chains   15.0 / 11.5
                                  700 x 200, 1000 chains  38.9 / 20.2
                       linear     1024 x 64, 512 chains   11.1 / 13.9
                                  2048 x 64, 256 chains    9.1 / 13.6
                                  3000 x 8,  64 chains    12.5 / 10.1
              float64  logistic   512 x 64,  256 chains    8.0 / 16.2
                                  1024 x 64, 256 chains   13.6 / 16.7
                                  1024 x 30, 512 chains   15.9 / 14.4
                                  1024 x 100, 64 chains   23.8 / 15.6
                       linear     2048 x 30, 64 chains     9.5 / 11.6
                                  3000 x 30, 64 chains    13.0 / 11.9
  batch       float32  logistic   16 of 128..600 x 30, 16 chains    16.6 / 21.4
              float64  logistic   256 of 512..2000 x 4, 1 chain     41.0 / 78.7

In float64 a logistic density's exponentials make the per-chain pass up to
three times as dear as a linear one's, so some lines hold for logistic ones
only.
"""

import numpy as np
import torch

from probability_amd import _lib
from probability_amd import tuning

_REGRESSIONS = (_lib.TARGET_LOGISTIC, _lib.TARGET_LINEAR)


def max_columns(dtype):
  """The most coefficients the tiles hold."""
  return 256 if dtype == torch.float32 else 128


def takes_eval(spec, dim, chains):
  """Whether log densities and gradients of `chains` chains of a spec of state
  size `dim` are tiled."""
  kind = spec.kind
  if kind not in _REGRESSIONS or chains < 1:
    return False
  n, d = spec.base.n_obs, dim - (kind == _lib.TARGET_LINEAR)
  if d > max_columns(spec.dtype):
    return False
  if chains >= 4096:
    return n >= 512
  if spec.dtype == torch.float32:
    return n >= (900 if d >= 64 else 1200) or n * d >= 110000
  if kind == _lib.TARGET_LOGISTIC:
    return n >= 900 or n * d >= 27000
  return n >= 1400 or n * d >= 70000


# How long the per-chain path's leapfrog is, in passes of a wave over its
# registers' worth of rows, from where trajectories are tiled: per (float32,
# logistic) the columns up to which a line holds, the passes, and the same for
# trajectories of one or two steps, which carry the launch that starts them.
_PASSES = {
    (True, True): ((128, 3.0, 4.0), (256, 0.0, 0.0)),
    (True, False): ((16, 3.0, 3.4), (32, 2.2, 0.0), (64, 3.4, 3.4),
                    (128, 2.2, 0.0), (256, 0.0, 0.0)),
    (False, True): ((16, 3.2, 0.0), (32, 0.0, 0.0), (64, 2.5, 2.5),
                    (128, 1.2, 0.0)),
    (False, False): ((16, 2.5, 0.0), (32, 3.2, 0.0), (64, 4.5, 0.0),
                     (128, 0.0, 0.0)),
}


def takes_trajectory(spec, dim, chains, leapfrogs):
  """Whether HMC trajectories of `chains` chains are tiled: from the rows and
  chains on that are worth the launches of trajectories, and where the
  per-chain path takes more than a few passes.  Its waves share a chain's
  rows (256 a pass, 128 of float64 rows of more than 32 columns); more waves
  than the 1024 that run at once take proportionally longer in float64, which
  is bound by arithmetic, and less in float32."""
  kind = spec.kind
  if kind not in _REGRESSIONS or chains < 1 or leapfrogs < 1:
    return False
  n, d = spec.base.n_obs, dim - (kind == _lib.TARGET_LINEAR)
  if d > max_columns(spec.dtype):
    return False
  f = 1 if leapfrogs > 2 else 2
  f32, logistic = spec.dtype == torch.float32, kind == _lib.TARGET_LOGISTIC
  if f32:
    long = n >= 3000 * f or (
        n >= 512 and n * chains >= (500000 if n >= 700 else 700000) * f)
  elif d >= 64 and logistic:
    long = n >= 1024 * f or n * chains >= 131072 * f
  else:
    long = n >= 2048 * f or (
        n >= 512 and n * chains >= (500000 if d > 16 else 1000000) * f)
  if not long:
    return False
  waves = min(4, tuning.glm_waves(kind, n, dim, chains, 'hmc', spec.dtype))
  passes = -(-n // ((256 if f32 or d <= 32 else 128) * waves))
  passes *= max(1.0, chains * waves / 1024) ** (0.6 if f32 else 1.0)
  least = next(v for v in _PASSES[f32, logistic] if d <= v[0])
  return passes >= least[f]


def dim_x(spec):
  """Coefficients of a regression spec (or of the one it transforms)."""
  return spec.dim - (spec.kind == _lib.TARGET_LINEAR)


def plan(spec, chains, dim_stride, trajectory):
  p = _lib.GlmPlan()
  _lib.check(_lib.lib().hipmc_glm_tile_plan(
      _lib.dtype_code(spec.dtype), spec.base.n_obs, dim_x(spec), chains,
      dim_stride, 1 if trajectory else 0, p))
  return p


def _workspace(p, device):
  return torch.empty(p.workspace_bytes, dtype=torch.uint8, device=device)


def evaluate(spec, table, x, tlp, grad):
  """Log density [C] and gradient [C, stride] of `spec` at x [C, stride]."""
  c, stride = x.shape
  ws = _workspace(plan(spec, c, stride, False), x.device)
  _lib.check(_lib.lib().hipmc_glm_tile_eval(
      _lib.dtype_code(spec.dtype), _lib.ptr(table), spec.base.n_obs,
      dim_x(spec), spec.dim, c, stride, _lib.ptr(x), _lib.ptr(tlp),
      _lib.ptr(grad), _lib.ptr(ws), ws.numel(),
      _lib.stream_handle(x.device)))


def run_hmc(spec, args, calibrated, device):
  """hipmc_hmc_run (calibrated) or hipmc_leapfrog_run on the tiles."""
  ws = _workspace(plan(spec, args.n_chains, args.dim_stride, True), device)
  _lib.check(_lib.lib().hipmc_glm_tile_hmc_run(
      args, 1 if calibrated else 0, spec.base.n_obs, dim_x(spec),
      _lib.ptr(ws), ws.numel(), _lib.stream_handle(device)))


class BatchTiles:
  """Tiles of a batch of regressions: chains of one problem by 32 (16 where
  no problem has more, or the columns are many), rows in ranges such that at
  most about 768 blocks run in all.  `table` is None where the batch is not
  tiled."""

  def __init__(self, rows, cols, chains, offsets, dtype, device):
    """Of problems with rows[i] observations, at most `cols` coefficients and
    chains[i] chains from row offsets[i]."""
    self.table = None
    rows, chains = np.asarray(rows), np.asarray(chains)
    n, c = int(rows.max()), int(chains.sum())
    if cols > max_columns(dtype) or n < 512 or chains.min() < 1:
      return
    # the per-chain pass takes as long as the longest problem's rows, until
    # the chains fill the GPU
    if c < 4096 and n < 1300 and n * cols < (
        110000 if dtype == torch.float32 else 70000):
      return
    slabs = -(-cols // 16)
    wide = slabs <= (8 if dtype == torch.float32 else 4)
    ct = 32 if wide and chains.max() > 16 else 16
    tiles = -(-chains // ct)
    n_tiles = int(tiles.sum())
    # many tiles of a few chains each are mostly empty (a narrow float64
    # design's per-chain pass is the cheaper: 512 of 128..4000 x 4, 8 chains 183
    # us, tiled 214)
    fill = 0.75 * ct if dtype == torch.float64 and cols <= 16 else 8
    if n_tiles > 128 and c < fill * n_tiles:
      return
    # rows per range, a multiple of 64: sum of tiles * ceil(rows / per) is at
    # most the sum of tiles * rows over per, plus the tiles
    per = -(-int((tiles * rows).sum()) // (64 * max(768 - n_tiles, 1))) * 64
    per = min(per, -(-int(rows.max()) // 64) * 64)
    prob = np.repeat(np.arange(len(rows)), tiles)
    first = (np.arange(n_tiles) - (np.cumsum(tiles) - tiles)[prob]) * ct
    splits = (-(-rows // per))[prob]
    ends = np.cumsum(splits)
    out = np.zeros((n_tiles, 8), np.int32)
    out[:, 0] = prob
    out[:, 1] = np.asarray(offsets)[prob] + first
    out[:, 2] = np.minimum(ct, chains[prob] - first)
    out[:, 3] = splits
    out[:, 4] = ends - splits
    out[:, 5] = per
    self.tile_chains, self.width, self.n_tiles = ct, 16 * slabs, n_tiles
    self.max_split, self.slots = int(splits.max()), int(ends[-1])
    self.table = torch.from_numpy(out).to(device)

  def evaluate(self, batch, x, tlp, grad):
    ws = torch.empty((self.slots, self.tile_chains, self.width),
                     dtype=batch.dtype, device=x.device)
    sums = torch.empty((self.slots, self.tile_chains), dtype=torch.float64,
                       device=x.device)
    _lib.check(_lib.lib().hipmc_glm_tile_eval_batch(
        _lib.dtype_code(batch.dtype), _lib.ptr(batch.table),
        _lib.ptr(self.table), self.n_tiles, self.max_split, self.slots,
        self.tile_chains, self.width, batch.max_dim, batch.dim_stride,
        _lib.ptr(x), _lib.ptr(tlp), _lib.ptr(grad), _lib.ptr(ws),
        _lib.ptr(sums), _lib.stream_handle(x.device)))
