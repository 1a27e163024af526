"""The hierarchical normal's specialised NUTS leaf (Softplus on the scale, no
momentum precision, register slots full but for the last) against the general
one, which a momentum precision of ones selects: multiplying by one changes
nothing, so every output but the energy (which then holds the momentum
density's constant) is the same bit for bit.  State sizes at the edges of the
register slots, both dtypes, trees up to depth 7."""

import numpy as np
import pytest
import torch

from probability_amd import _lib
from probability_amd import bijectors as bij
from probability_amd import targets as ptg
from probability_amd.mcmc import _runner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('groups', [1, 62, 63, 126, 127, 190, 191, 254, 255,
                                    318, 319])
def test_specialised_leaf_equals_general(groups, dtype):
  g = torch.Generator(device='cuda').manual_seed(groups)
  r = lambda *s: torch.randn(s, generator=g, device='cuda', dtype=dtype)
  spec = ptg.TransformedTarget(
      ptg.HierarchicalNormal(3 + 4 * r(groups), 8 + 4 * r(groups).abs(),
                             dtype=dtype),
      [bij.Identity(), bij.Softplus(), bij.Identity()])
  chains = 9
  x = 0.5 * r(chains, groups + 2)
  tlp, grad = spec.log_prob_and_grad_flat(x)
  step = torch.full((1,), 0.15, device='cuda', dtype=dtype)
  ones = torch.ones((1, groups + 2), device='cuda', dtype=dtype)
  out = []
  for precision in (None, ones):
    state, t, gr = x.clone(), tlp.clone(), grad.clone()
    run = _runner.Run(spec, spec.table(), state, t, gr, step,
                      np.array([7, groups], np.uint32), n_iters=3,
                      fold_seed=True)
    run.args.max_tree_depth = 7
    run.args.unrolled_leapfrog_steps = 1
    if precision is not None:
      run.args.momentum_precision = precision.data_ptr()
    o = [run.want('out_log_accept_ratio', (3, chains), dtype),
         run.want('out_leapfrogs', (3, chains), torch.int32),
         run.want('out_is_accepted', (3, chains), torch.bool)]
    run.call(_lib.lib().hipmc_nuts_run)
    out.append([state, t, gr] + o)
  assert int(out[0][4].max()) > 7
  for a, b in zip(*out):
    assert torch.equal(a, b)
