"""A batch that is dropped while another stream's launch still reads its
device arrays keeps their memory from the allocator until that work is done."""

import numpy as np
import pytest
import torch

from probability_amd import targets as ptg
from probability_amd.mcmc import batched

pytestmark = pytest.mark.gpu


def _arrays(batch):
  out = [batch.table, batch.chain_problem, batch.chain_local,
         batch.group_start]
  if batch._order is not None and batch._order[0] is not None:
    out.append(batch._order[0])
  if batch._tiles is not None and batch._tiles.table is not None:
    out.append(batch._tiles.table)
  return out


def _use(batch, use, x):
  if use == 'bijector':
    return batch.bijector(x, 0)
  if use == 'order':
    return batch.start_order().clone()
  return getattr(batch, use)(x)


@pytest.mark.parametrize('use', ['eval', 'eval_chains', 'bijector', 'order'])
def test_arrays_outlive_another_streams_work(use):
  r = np.random.default_rng(0)
  specs = []
  for n, d in ((600, 3), (2000, 9)):
    x = r.normal(size=(n, d)).astype(np.float32)
    specs.append(ptg.LogisticRegression(
        x, (r.uniform(size=n) < 0.5).astype(np.float32), device='cuda'))
  warm, batch = [batched.PosteriorBatch(specs, num_chains=4, waves_per_chain=4)
                 for _ in range(2)]
  x = torch.zeros((8, batch.dim_stride), device='cuda')
  order_on, side = torch.cuda.Stream(), torch.cuda.Stream()
  with torch.cuda.stream(side):  # whatever the first call of a kind loads
    torch.cuda._sleep(1000)
    _use(warm, use, x)
  if use == 'order':  # allocated on a run's stream, read on another run's
    with torch.cuda.stream(order_on):
      assert batch.start_order() is not None
  batch.eval(x)
  torch.cuda.synchronize()
  with torch.cuda.stream(side):
    torch.cuda._sleep(400_000_000)  # some 0.2 s
    got = _use(batch, use, x)
  sizes = [(t.data_ptr(), t.nbytes) for t in _arrays(batch)]
  del batch
  taken, held = set(), []
  for s in (torch.cuda.default_stream(), order_on):
    with torch.cuda.stream(s):
      for _, n in sizes:
        for _ in range(8):
          held.append(torch.empty(n, dtype=torch.uint8, device='cuda'))
          taken.add(held[-1].data_ptr())
  busy = not side.query()  # the launch above was still waiting
  torch.cuda.synchronize()
  assert busy
  assert not taken & {p for p, _ in sizes}
  del got
