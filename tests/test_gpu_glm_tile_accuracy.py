"""The tiled GLM gradient is no less exact than the per-chain pass.

Gradients of chains near the mode of a linear model, where residuals are small
differences of the logits, so that the logits' rounding shows.  The reference
is extended precision (80-bit; 2^-64, 2000 times finer than float64) for
float64 and float64 for float32.  The bound is the per-chain pass's own root
mean square error on the same inputs over three data sets: both kernels add
the same products, and what is held is that the tiles' order of additions
loses no more."""

import numpy as np
import pytest
import torch

from probability_amd import glm_tile
from probability_amd import targets as ptg

pytestmark = pytest.mark.gpu


def _squared_errors(n, d, c, ndt, seed):
  """Mean squared gradient errors, per-chain and tiled, over the largest
  gradient element."""
  wide = np.longdouble if ndt == np.float64 else np.float64
  r = np.random.default_rng([n, d, seed])
  x = r.normal(size=(n, d)).astype(ndt)
  y = (x @ (r.normal(size=d) / np.sqrt(d)) + 0.3 * r.normal(size=n)).astype(ndt)
  mode = np.linalg.lstsq(x.astype(np.float64), y.astype(np.float64),
                         rcond=None)[0]
  q = (mode + 0.01 / np.sqrt(n) * r.normal(size=(c, d))).astype(ndt)
  q = np.concatenate([q, np.full((c, 1), 0.3, ndt)], 1)
  xw, qw = x.astype(wide), q.astype(wide)
  res = y.astype(wide)[:, None] - xw @ qw[:, :d].T
  want = (xw.T @ res).T / qw[:, d:] ** 2 - qw[:, :d]
  spec = ptg.LinearRegression(
      x, y, dtype=torch.float64 if ndt == np.float64 else torch.float32,
      device='cuda')
  t = torch.as_tensor(q, device='cuda')
  tlp, tiled = torch.empty_like(t[:, 0]), torch.empty_like(t)
  glm_tile.evaluate(spec, spec.table(), t, tlp, tiled)
  _, chain = spec.log_prob_and_grad_chains(t)
  scale = np.abs(want).max()
  return [float((((g.cpu().numpy()[:, :d].astype(wide) - want) / scale) ** 2
                 ).mean()) for g in (chain, tiled)]


@pytest.mark.parametrize('ndt', [np.float32, np.float64])
@pytest.mark.parametrize('n,d,c', [
    (1500, 16, 40), (1501, 30, 64), (1024, 64, 12), (2000, 64, 40),
    (1024, 80, 16), (1300, 96, 20), (1024, 112, 16), (1024, 127, 30),
    (4100, 128, 16)])
def test_gradient_error_is_no_larger_than_the_per_chain_pass(n, d, c, ndt):
  chain, tiled = np.sum([_squared_errors(n, d, c, ndt, s) for s in range(3)], 0)
  print(f'rms error {chain ** 0.5:.3g} -> {tiled ** 0.5:.3g}, '
        f'ratio {(tiled / chain) ** 0.5:.3f}')
  assert tiled <= chain
