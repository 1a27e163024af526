"""The per-chain step of the BF16 MFMA path at the row-split counts where its
reduction changes form (whole batches of 32 and 8 splits, remainders, more
than one 64-lane group of log-likelihoods), against the float64 oracle on the
same BF16-rounded X.  Tolerances as in test_gpu_mfma.py: 1e-5 normwise
(BF16 hi/lo products, FP32 sums), 1e-3 on log accept ratios."""

import numpy as np
import pytest
import torch

from oracle import mcmc as omcmc
from oracle import rng as orng
from oracle import targets as otg
from probability_amd import targets as ptg
from probability_amd.mcmc import glm_mfma

pytestmark = pytest.mark.gpu


def _normwise(got, want, tol):
  got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
  assert np.abs(got - want).max() <= tol * max(np.abs(want).max(), 1.0)


@pytest.mark.parametrize('splits', [1, 7, 8, 33, 41, 64, 70])
def test_chain_step_over_split_counts_matches_oracle(splits):
  n, c, steps, eps = 32 * splits, 64, 3, np.float32(0.02)
  r = np.random.default_rng(splits)
  x = (r.normal(size=(n, 256)) / 16).astype(np.float32)
  beta = r.normal(size=256)
  y = (r.uniform(size=n) < 1 / (1 + np.exp(-(x @ beta)))).astype(np.float32)
  spec = ptg.LogisticRegressionBF16(x, y)
  o = otg.LogisticRegression(spec.x.double().cpu().numpy(),
                             y.astype(np.float64))
  q = (r.normal(size=(c, 256)) * 0.3).astype(np.float32)
  runner = glm_mfma.GlmHmcRunner(spec, c, n_split=splits)
  state = torch.as_tensor(q, device='cuda')
  tlp, grad = runner.bootstrap(state)
  t0, g0 = o.log_prob_and_grad(q.astype(np.float64))
  _normwise(tlp.cpu().numpy(), t0, 1e-5)
  _normwise(grad.cpu().numpy(), g0, 1e-5)
  seed = orng.sanitize_seed(splits)
  lar = torch.empty((1, c), device='cuda')
  acc = torch.empty((1, c), dtype=torch.uint8, device='cuda')
  trace = torch.empty((1, c, 256), device='cuda')
  step = torch.full((1,), float(eps), device='cuda')
  runner.run(state, tlp, grad, step, seed, steps, out_lar=lar, out_acc=acc,
             trace=trace, n_trace=1)
  oq, ores = omcmc.hmc_one_step(o, eps, steps, q.astype(np.float64), t0, g0,
                                seed, orng.PhiloxDraws(np.float32))
  np.testing.assert_allclose(lar[0].cpu().numpy(), ores.log_accept_ratio,
                             atol=1e-3, rtol=0)
  got = acc[0].cpu().numpy().astype(bool)
  u = orng.mh_uniform(orng.split_seed(seed, 2)[1], np.arange(c), np.float32)
  clear = np.abs(np.log(u.astype(np.float64)) - ores.log_accept_ratio) > 1e-3
  np.testing.assert_array_equal(got[clear], ores.is_accepted[clear])
  same = got == ores.is_accepted
  _normwise(state.cpu().numpy()[same], oq[same], 1e-5)
  assert torch.equal(trace[0], state)
