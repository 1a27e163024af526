"""Batches whose specs are themselves transformed, once or twice: they run
with the caller's waves per chain and draw what the plain specs draw (the
batch's own bijectors say how the state is transformed)."""

import numpy as np
import pytest
import torch

from probability_amd import bijectors as pbij
from probability_amd import targets as ptg
from probability_amd.mcmc import batched

pytestmark = pytest.mark.gpu


def _specs():
  r = np.random.default_rng(0)
  out = []
  for n, d in ((60, 3), (700, 5)):
    x = r.normal(size=(n, d)).astype(np.float32)
    y = (r.uniform(size=n) < 0.5).astype(np.float32)
    out.append(ptg.LogisticRegression(x, y, device='cuda'))
  return out


@pytest.mark.parametrize('layers', [1, 2])
@pytest.mark.parametrize('kernel', ['nuts', 'hmc'])
def test_transformed_specs_draw_what_plain_ones_draw(kernel, layers):
  plain = _specs()
  wrapped = list(plain)
  for _ in range(layers):
    wrapped = [ptg.TransformedTarget(s, [pbij.Identity()]) for s in wrapped]
  draws = []
  for specs in (plain, wrapped):
    batch = batched.PosteriorBatch(specs, num_chains=4, waves_per_chain=2)
    x = torch.zeros((8, batch.dim_stride), device='cuda')
    tlp, grad = batch.eval(x)
    res = batched.sample_posteriors(batch, 3, step_size=0.05, kernel=kernel,
                                    seed=[1, 2])
    draws.append([tlp, grad] + list(res.draws))
  for a, b in zip(*draws):
    assert torch.equal(a, b)
