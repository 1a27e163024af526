"""Float64 regressions' NUTS chains from the queue have a kernel of their own:
their draws equal, bit for bit, those of the problem alone, whose launch fits
the GPU and takes the other kernel.  One size per register slot count, both
models, each number of waves that share a chain."""

import numpy as np
import pytest
import torch

from probability_amd import bijectors as pbij
from probability_amd import targets as ptg
from probability_amd.mcmc import batched

pytestmark = pytest.mark.gpu


def _spec(model, n, d, seed):
  r = np.random.default_rng([n, d, seed])
  x = r.normal(size=(n, d))
  s = x @ r.normal(size=d) / np.sqrt(d)
  if model == 'logistic':
    y = (r.uniform(size=n) < 1 / (1 + np.exp(-s))).astype(np.float64)
    return ptg.LogisticRegression(x, y, dtype=torch.float64), [pbij.Identity()]
  return (ptg.LinearRegression(x, s + 0.5 * r.normal(size=n),
                               dtype=torch.float64),
          [pbij.Identity(), pbij.Exp()])


def _run(cases, chains, keys, waves, slot_dim):
  batch = batched.PosteriorBatch(
      [s for s, _ in cases], chains, bijectors=[b for _, b in cases],
      keys=keys, slot_dim=slot_dim, waves_per_chain=waves)
  return batched.sample_posteriors(
      batch, 2, num_burnin_steps=1, step_size=0.03, max_tree_depth=4, seed=5)


@pytest.mark.parametrize('waves', [2, 8])
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('d', [40, 100, 170, 230, 300, 400])
def test_queued_draws_equal_the_problems_alone(d, model, waves):
  cases = [_spec(model, n, d - 7 * i, i) for i, n in enumerate((50, 130, 77))]
  chains = 8 // waves * 256 // 3 + 40  # more than fit at once, in all
  both = _run(cases, chains, [0, 1, 2], waves, d + 1)
  for i, case in enumerate(cases):
    alone = _run([case], chains, [i], waves, d + 1)
    assert torch.equal(both.draws[i], alone.draws[0])
    assert torch.equal(both.leapfrogs_taken[i], alone.leapfrogs_taken[0])
    assert bool(torch.isfinite(alone.draws[0]).all())
