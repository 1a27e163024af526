"""ESS and R-hat calls that the device kernels leave to the torch form give
what the kernels give for the same question asked in a form they take."""

import numpy as np
import pytest
import torch

from probability_amd.mcmc import diagnostic as pdiag

pytestmark = pytest.mark.gpu


def _draws(n, c, d, seed=0, dtype=np.float32):
  r = np.random.default_rng(seed)
  x = r.normal(size=(n, c, d))
  for t in range(1, n):
    x[t] = 0.6 * x[t - 1] + 0.8 * x[t]
  return torch.as_tensor((x + 3).astype(dtype), device='cuda')


@pytest.mark.parametrize('where', ['cuda', 'cpu one element', 'float32'])
def test_threshold_tensors_broadcast_over_the_dimensions(where):
  x = _draws(200, 6, 3)
  th = [0.0, 0.1, 0.3]
  if where == 'cuda':
    arg = torch.tensor(th, dtype=torch.float64, device='cuda')
  elif where == 'float32':
    arg = torch.tensor([0.25, 0.5, 0.125], device='cuda')
    th = [0.25, 0.5, 0.125]
  else:
    arg, th = torch.tensor(0.1, dtype=torch.float64), [0.1] * 3
  got = pdiag.effective_sample_size(x, filter_threshold=arg,
                                    cross_chain_dims=1)
  want = torch.stack([
      pdiag.effective_sample_size(x, filter_threshold=t, cross_chain_dims=1)[i]
      for i, t in enumerate(th)])
  # the forms' transforms differ by rounding (see the size tests' bound)
  torch.testing.assert_close(got, want, rtol=1e-9, atol=0)


def test_ess_rule_and_limits():
  takes = pdiag._ess_takes
  assert takes(1, 2, 1) and takes(4096, 2, 1) and not takes(4097, 2, 1)
  assert not takes(100, 1, 5) and not takes(100, 1 << 29, 2)
  assert takes(8, 2, 25000) and not takes(8, 2, 25001) and takes(9, 2, 25001)
  assert takes(64, 65536, 1) and not takes(64, 65537, 1) and takes(65, 65537, 1)
  assert takes(4096, 2, (1 << 22) - 1) and not takes(4096, 2, 1 << 22)


@pytest.mark.parametrize('n,c,d', [(4, 2, 25001), (8, 7000, 9), (8, 2, 25000),
                                   (9, 2, 30000), (64, 70000, 1), (70, 70000, 1)])
def test_ess_on_both_sides_of_the_rule(n, c, d):
  """Against the same draws in float64 on the CPU, which the kernels never
  take (tolerance as above)."""
  x = _draws(n, c, d, n)
  want = pdiag.effective_sample_size(x.double().cpu(), cross_chain_dims=1,
                                     filter_threshold=None)
  got = pdiag.effective_sample_size(x, cross_chain_dims=1,
                                    filter_threshold=None)
  torch.testing.assert_close(1 / got.cpu(), 1 / want, rtol=1e-9, atol=1e-12)
