"""R-hat keeps float64's precision where a few draws lie far from the rest.

The reference is the formula in 80-bit arithmetic, two passes.  Tolerance 1e-13
relative: variances are sums of positive terms over groups of 16 draws, their
merges (at most some 64 in a row at these sizes) and as many merges of chains,
each of a few operations that round by 1.1e-16: below 3e-14, and R-hat is a
few operations on such variances."""

import numpy as np
import pytest
import torch

from probability_amd.mcmc import diagnostic as pdiag

pytestmark = pytest.mark.gpu


def _rhat(x, split):
  x = x.astype(np.longdouble)
  if split:
    h = x.shape[0] // 2
    x = np.concatenate([x[:h], x[h:2 * h]], 1)
  n, m = x.shape[:2]
  w = x.var(0, ddof=1).mean(0)
  s2 = (n - 1) * w / n + x.mean(0).var(0, ddof=1)
  return (m + 1) * s2 / (m * w) - np.longdouble(n - 1) / (m * n)


@pytest.mark.parametrize('split', [True, False])
@pytest.mark.parametrize('n,c,d', [(20000, 4, 3), (20000, 2, 1), (3001, 9, 70),
                                   (200001, 2, 2)])
@pytest.mark.parametrize('dtype', [np.float32, np.float64])
def test_an_outlying_first_draw_costs_no_precision(dtype, n, c, d, split):
  r = np.random.default_rng(n + c + d)
  # chains apart, so that R-hat is as exact as their variances
  x = r.normal(size=(n, c, d)) + 3 * r.normal(size=(c, 1))
  x[0] += 100       # where the chains start
  x[n // 2] += 100  # and the second half
  x = x.astype(dtype)
  got = pdiag.potential_scale_reduction(torch.as_tensor(x, device='cuda'),
                                        split_chains=split).cpu().numpy()
  want = _rhat(x, split)
  err = np.abs((got - want) / want).max()
  print(f'relative error {float(err):.2e}')
  assert err <= 1e-13


@pytest.mark.parametrize('value', [3.0, 0.1, 1e30])
@pytest.mark.parametrize('n,c,d', [(1000, 4, 3), (37, 300, 1)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
def test_chains_that_never_move_have_no_variance(dtype, n, c, d, value):
  x = torch.full((n, c, d), value, dtype=dtype, device='cuda')
  assert bool(torch.isnan(pdiag.potential_scale_reduction(
      x, split_chains=True)).all())
  x[:, 0] *= 2  # variance between the chains only
  assert bool(torch.isinf(pdiag.potential_scale_reduction(
      x, split_chains=True)).all())
