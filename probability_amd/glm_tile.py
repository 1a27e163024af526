"""When a regression's chains take the tiled evaluation (csrc/glm_tile.h: the
logits and gradients of many chains as matrix products over row ranges), and
its workspaces.

The other path is the sampling kernels' own: one chain per wave (up to four
waves per chain in HMC) passing over X by itself, one launch for a whole
trajectory.  The tiled one pays two launches per gradient, about 9 to 13 us
however small the problem.  Where the lines lie, us per evaluation (or per
leapfrog step) one chain per wave / tiled, logistic regression, MI355X:

  evaluation  float32  256 x 100, 512 chains   11.1 / 13.1
                       512 x 6,   64 chains    10.7 / 10.1
                       512 x 30,  512 chains   13.6 / 9.7
                       8192 x 100, 8 chains     212 / 12
              float64  256 x 30,  512 chains   10.5 / 12.3
                       128 x 100, 64 chains    14.8 / 13.0
  trajectory  float32  2048 x 6,  64 chains     9.9 / 10.6
                       4096 x 6,  64 chains    17.4 / 11.3
                       512 x 30,  512 chains   11.3 / 11.4
                       1024 x 30, 512 chains   20.7 / 11.8
                       512 x 30,  2048 chains  22.6 / 12.6
              float64  1024 x 6,  512 chains   12.7 / 13.9
                       2048 x 6,  64 chains    20.9 / 12.7
                       1024 x 30, 512 chains   19.3 / 15.0
                       256 x 100, 64 chains    14.5 / 14.4
                       256 x 100, 512 chains   29.5 / 15.0

In float64 a logistic density's exponentials make the per-chain pass up to
three times as dear as a linear one's (128 x 100, 64 chains, evaluation
14.8 against 11.6; 1024 x 64, 8 chains, trajectory 24.9 against 9.5), so the
lines of narrow or short designs hold for logistic ones only.
"""

import numpy as np
import torch

from probability_amd import _lib

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
  return n >= 512 or (spec.dtype == torch.float64 and n * d >= 12000 and
                      kind == _lib.TARGET_LOGISTIC)


def takes_trajectory(spec, dim, chains, leapfrogs):
  """Whether HMC trajectories of `chains` chains are tiled.  Trajectories of
  one or two steps carry the launch that starts them as well."""
  kind = spec.kind
  if kind not in _REGRESSIONS or chains < 1 or leapfrogs < 1:
    return False
  n, d = spec.base.n_obs, dim - (kind == _lib.TARGET_LINEAR)
  if d > max_columns(spec.dtype):
    return False
  f = 1 if leapfrogs > 2 else 2
  if spec.dtype == torch.float32:
    return n >= 3000 * f or (n >= 512 and n * chains >= 500000 * f)
  if n >= 2048 * f:
    return True
  if d >= 64 and kind == _lib.TARGET_LOGISTIC:
    return n >= 1024 * f or n * chains >= 131072 * f
  return n >= 512 and n * chains >= (500000 if d > 16 else 1000000) * f


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
    if (cols > max_columns(dtype) or rows.max() < 512 or chains.min() < 1):
      return
    slabs = -(-cols // 16)
    wide = slabs <= (8 if dtype == torch.float32 else 4)
    ct = 32 if wide and chains.max() > 16 else 16
    tiles = -(-chains // ct)
    n_tiles = int(tiles.sum())
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
