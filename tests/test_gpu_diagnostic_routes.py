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
