"""The per-chain pass and the per-chain trajectory kernel at the sizes that
the public calls send to the tiles: they start every batched and serving run,
and run what the tiles do not hold.  The oracle checks and tolerances of the
public calls."""

import numpy as np
import pytest
import torch

import test_gpu_parity as parity
from oracle import mcmc as omcmc
from oracle import rng as orng
from probability_amd import _lib
from probability_amd.mcmc import _runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('tdt,ndt,tol', parity.DTYPES)
@pytest.mark.parametrize('kind', ['logistic', 'linear', 'logistic_split',
                                  'linear_split', 'logistic_wide',
                                  'logistic_d150', 'linear_wide',
                                  'logistic_tall'])
def test_per_chain_evaluation_matches_oracle(kind, tdt, ndt, tol):
  o, mk, q, codes = parity._case(kind, ndt)
  spec = mk(tdt)
  x = torch.as_tensor(q, dtype=tdt, device='cuda')
  tlp, grad = spec.log_prob_and_grad_chains(x, parity._bijs(spec, codes))
  rt, rg = parity._otarget(o, codes).log_prob_and_grad(q)
  parity._check(f'chains {kind} tlp', parity._np(tlp), rt, tol)
  parity._check(f'chains {kind} grad', parity._np(grad), rg, tol)


@pytest.mark.parametrize('tdt,ndt,tol', parity.DTYPES)
@pytest.mark.parametrize('kind,eps,steps', [
    ('logistic_split', 0.05, 8), ('logistic_wide', 0.02, 8),
    ('logistic_tall', 0.02, 5)])
@pytest.mark.parametrize('waves', [1, 2, 4])
def test_per_chain_trajectory_matches_oracle(kind, eps, steps, waves, tdt, ndt,
                                             tol):
  o, mk, q, _ = parity._case(kind, ndt, seed=3)
  spec = mk(tdt)
  x = torch.as_tensor(q, dtype=tdt, device='cuda')
  tlp, grad = spec.log_prob_and_grad_chains(x)
  seed = orng.sanitize_seed(77)
  run = _runner.Run(spec, spec.table(), x, tlp, grad,
                    torch.full((1,), eps, dtype=tdt, device='cuda'), seed,
                    sampler='hmc')
  run.args.num_leapfrog_steps, run.args.waves_per_chain = steps, waves
  c, d = q.shape
  lar = run.want('out_log_accept_ratio', (1, c), tdt)
  acc = run.want('out_is_accepted', (1, c), torch.bool)
  prop = run.want('out_proposed_state', (c, d), tdt)
  run.call(_lib.lib().hipmc_hmc_run)
  t0, g0 = o.log_prob_and_grad(q)
  oq, ores = omcmc.hmc_one_step(o, np.asarray(eps, ndt), steps, q, t0, g0,
                                seed, orng.PhiloxDraws(ndt))
  np.testing.assert_array_equal(parity._np(acc[0]), ores.is_accepted)
  parity._check(f'{kind} state', parity._np(x), oq, tol)
  parity._check(f'{kind} proposed', parity._np(prop), ores.proposed_state, tol)
  parity._check(f'{kind} lar', parity._np(lar[0]), ores.log_accept_ratio, tol,
                scale=np.abs(t0).max())
