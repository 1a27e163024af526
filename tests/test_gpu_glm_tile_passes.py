"""The tiled GLM evaluation where a block makes several passes over its rows:
the next rows' loads in flight, the staged rows overwritten, sums carried from
pass to pass, a ragged last pass.  Same oracle and tolerances as at the edges
of the tiles."""

import numpy as np
import pytest

import test_gpu_glm_tile as tiles
from oracle import mcmc as omcmc
from oracle import rng as orng
from probability_amd import glm_tile

pytestmark = pytest.mark.gpu

# (rows, columns, chains); float64 holds at most 128 columns
SHAPES = [(1100, 20, 1000), (2100, 100, 500), (1500, 3, 2100), (3333, 64, 700),
          (1500, 250, 700), (1300, 113, 1100)]


def _passes(spec, c, trajectory):
  """At least three passes in every range, the last one short."""
  p = glm_tile.plan(spec, c, spec.dim, trajectory)
  n = spec.base.n_obs
  assert p.rows_per_split >= 3 * 64 and p.n_split > 1
  last = n - (p.n_split - 1) * p.rows_per_split
  assert last > 64 and last % 16 != 0


@pytest.mark.parametrize('tdt,ndt,tol', tiles.TYPES)
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('n,d,c', SHAPES)
def test_density_and_gradient_match_oracle(n, d, c, model, tdt, ndt, tol):
  if d > glm_tile.max_columns(tdt):
    d = glm_tile.max_columns(tdt)
  spec, o, q = tiles._case(model, n, d, c, ndt, n + d)
  _passes(spec, c, False)
  t, g = o.log_prob_and_grad(q.astype(np.float64))
  tlp, grad = tiles._evaluate(spec, q)
  tiles._normwise(tlp, t, tol)
  tiles._normwise(grad, g, tol)


@pytest.mark.parametrize('tdt,ndt,tol', tiles.TYPES)
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('n,d,c,steps', [(1100, 20, 1000, 2),
                                         (2100, 100, 500, 3)])
def test_trajectories_match_oracle(n, d, c, steps, model, tdt, ndt, tol):
  spec, o, q = tiles._case(model, n, d, c, ndt, n)
  _passes(spec, c, True)
  eps, seed = ndt(0.005), orng.sanitize_seed(n)
  x, t, g, p0, p1, _ = tiles._leapfrog(spec, q, eps, steps, seed)
  qd = q.astype(np.float64)
  t0, g0 = o.log_prob_and_grad(qd)
  want0 = orng.PhiloxDraws(ndt).momentum(seed, c, spec.dim).astype(np.float64)
  w1, wq, wt, wg = omcmc.leapfrog(o, float(eps), steps, want0, qd, t0, g0)
  for got, want in ((p0, want0), (x, wq), (t, wt), (g, wg), (p1, w1)):
    tiles._normwise(got, want, tol)
