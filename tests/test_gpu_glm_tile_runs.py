"""HMC, MALA and sample_chain over regressions large enough that the public
calls take the tiled trajectories: one transition against the oracle, the
fused run against the host step loop.  Each test checks that the tiles are
what ran.  Tolerances: states and densities of one transition 1e-5 / 1e-11
normwise, acceptance ratios (differences of densities) relative to the
densities; a fused run and a step loop are the same launches, so equal."""

import numpy as np
import pytest
import torch

import test_gpu_glm_tile as tiles
from oracle import mcmc as omcmc
from oracle import rng as orng
from probability_amd import glm_tile
from probability_amd import mcmc

pytestmark = pytest.mark.gpu

# model, rows, columns, chains: past the lines of both types for trajectories
# of three steps, and (the last two) of one
CASES = [('logistic', 3100, 6, 40), ('linear', 6100, 30, 12),
         ('logistic', 700, 6, 2400), ('logistic', 6200, 9, 33),
         ('linear', 8200, 20, 5)]


@pytest.fixture
def runs(monkeypatch):
  """Counts the calls of the tiled trajectories."""
  seen = []
  inner = glm_tile.run_hmc
  monkeypatch.setattr(glm_tile, 'run_hmc',
                      lambda *a: (seen.append(1), inner(*a))[1])
  return seen


def _state(spec, q):
  x = torch.as_tensor(q, device='cuda')
  return x, spec.unpack_state(x, (q.shape[0],))


def _step(n):
  return 0.3 / np.sqrt(n)


def _np(t):
  return t.detach().cpu().numpy()


@pytest.mark.parametrize('tdt,ndt,tol', tiles.TYPES)
@pytest.mark.parametrize('model,n,d,c', CASES)
def test_hmc_step_matches_oracle(model, n, d, c, tdt, ndt, tol, runs):
  if (model, n, ndt) == ('logistic', 700, np.float64):
    d, c = 100, 400  # the float64 line of short designs
  spec, o, q = tiles._case(model, n, d, c, ndt, n + d)
  eps, steps, seed = ndt(_step(n)), 3, orng.sanitize_seed(n)
  kernel = mcmc.HamiltonianMonteCarlo(spec, step_size=float(eps),
                                      num_leapfrog_steps=steps)
  x, parts = _state(spec, q)
  nxt, res = kernel.one_step(parts, kernel.bootstrap_results(parts), seed=seed)
  assert len(runs) == 1
  qd = q.astype(np.float64)
  t0, g0 = o.log_prob_and_grad(qd)
  oq, ores = omcmc.hmc_one_step(o, eps, steps, qd, t0, g0, seed,
                                orng.PhiloxDraws(ndt))
  np.testing.assert_array_equal(_np(res.is_accepted), ores.is_accepted)
  tiles._normwise(_np(spec.pack_state(nxt)), oq, tol)
  tiles._normwise(_np(spec.pack_state(res.proposed_state)),
                  ores.proposed_state, tol)
  scale = max(np.abs(t0).max(), 1.0)
  assert np.abs(_np(res.log_accept_ratio) - ores.log_accept_ratio).max() <= \
      tol * scale


@pytest.mark.parametrize('tdt,ndt,tol', tiles.TYPES)
@pytest.mark.parametrize('model,n,d,c', CASES[-2:])
def test_mala_step_matches_oracle(model, n, d, c, tdt, ndt, tol, runs):
  spec, o, q = tiles._case(model, n, d, c, ndt, n + d)
  eps, seed = ndt(0.2 / n), orng.sanitize_seed(n)
  kernel = mcmc.MetropolisAdjustedLangevinAlgorithm(spec, step_size=float(eps))
  x, parts = _state(spec, q)
  nxt, res = kernel.one_step(parts, kernel.bootstrap_results(parts), seed=seed)
  assert len(runs) == 1
  qd = q.astype(np.float64)
  t0, g0 = o.log_prob_and_grad(qd)
  oq, ores = omcmc.mala_one_step(o, eps, qd, t0, g0, seed,
                                 orng.PhiloxDraws(ndt))
  np.testing.assert_array_equal(_np(res.is_accepted), ores.is_accepted)
  tiles._normwise(_np(spec.pack_state(nxt)), oq, tol)
  tiles._normwise(_np(spec.pack_state(res.proposed_state)),
                  ores.proposed_state, tol)
  scale = max(np.abs(t0).max(), 1.0)
  assert np.abs(_np(res.log_accept_ratio) - ores.log_accept_ratio).max() <= \
      tol * scale


@pytest.mark.parametrize('tdt,ndt,tol', tiles.TYPES)
@pytest.mark.parametrize('adapt', [0, 4])
@pytest.mark.parametrize('model,n,d,c', CASES[:2])
def test_fused_run_equals_step_loop(model, n, d, c, adapt, tdt, ndt, tol,
                                    runs):
  spec, o, q = tiles._case(model, n, d, c, ndt, n + d)
  kernel = mcmc.HamiltonianMonteCarlo(spec, step_size=_step(n),
                                      num_leapfrog_steps=3)
  fields = ['log_accept_ratio', 'target_log_prob']
  if adapt:
    kernel = mcmc.DualAveragingStepSizeAdaptation(
        kernel, num_adaptation_steps=adapt, target_accept_prob=0.8)
    fields.append('step_size')
  x, parts = _state(spec, q)
  kw = dict(kernel=kernel, num_burnin_steps=5, num_steps_between_results=2,
            trace_fn=mcmc.TraceFields(*fields), seed=[3, n],
            return_final_kernel_results=False)
  a_states, a_trace = mcmc.sample_chain(4, parts, **kw)
  fused = len(runs)
  assert fused > 0
  b_states, b_trace = mcmc.sample_chain(4, parts, experimental_fused=False,
                                        **kw)
  assert len(runs) - fused == 5 + 1 + 3 * 3  # every step of the loop
  for u, v in list(zip(a_states, b_states)) + list(zip(a_trace, b_trace)):
    assert torch.equal(u, v)
  # the chains moved, and by accepted steps
  assert not torch.equal(a_states[0][0], a_states[0][-1])
