"""The BF16 MFMA gradient at the row-tile counts per split where its pipeline
has a different start or end (1 to 5 tiles of 32 rows, a shorter last split)
and at chain counts of both workgroup widths, against the float64 oracle on
the same BF16-rounded X.  Tolerance as in test_gpu_mfma.py: 1e-5 normwise
(BF16 hi/lo products, FP32 sums)."""

import numpy as np
import pytest
import torch

from oracle import targets as otg
from probability_amd import targets as ptg
from probability_amd.mcmc import glm_mfma

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('chains', [64, 128, 192])
@pytest.mark.parametrize('tiles,splits', [(1, 1), (2, 1), (3, 1), (4, 1),
                                          (5, 1), (5, 2), (8, 3), (13, 3)])
def test_gradient_over_tile_counts_matches_oracle(tiles, splits, chains):
  r = np.random.default_rng(100 * tiles + chains)
  n = 32 * tiles
  x = (r.normal(size=(n, 256)) / 16).astype(np.float32)
  beta = r.normal(size=256)
  y = (r.uniform(size=n) < 1 / (1 + np.exp(-(x @ beta)))).astype(np.float32)
  spec = ptg.LogisticRegressionBF16(x, y)
  o = otg.LogisticRegression(spec.x.double().cpu().numpy(),
                             y.astype(np.float64))
  q = (r.normal(size=(chains, 256)) * 0.3).astype(np.float32)
  runner = glm_mfma.GlmHmcRunner(spec, chains, n_split=splits)
  tlp, grad = runner.bootstrap(torch.as_tensor(q, device='cuda'))
  t0, g0 = o.log_prob_and_grad(q.astype(np.float64))
  for got, want in ((tlp, t0), (grad, g0)):
    got = got.double().cpu().numpy()
    assert np.abs(got - want).max() <= 1e-5 * max(np.abs(want).max(), 1.0)
