"""Launch helpers: build `hipmc_run_args` for a target spec and call libhipmc.

Single-problem launches use chain_problem = chain_local = NULL, so chain c's
draws are keyed (problem 0, chain c).
"""

import numpy as np
import torch

from probability_amd import _lib
from probability_amd import glm_tile
from probability_amd import targets as targets_lib
from probability_amd import tuning
from probability_amd.mcmc.internal import util as mcmc_util

_OUT_FIELDS = ('out_log_accept_ratio', 'out_leapfrogs', 'out_is_accepted',
               'out_reach_max_depth', 'out_has_divergence', 'out_energy',
               'out_tree_depth', 'trace_state', 'out_proposed_state',
               'out_proposed_tlp', 'out_initial_momentum',
               'out_final_momentum')


def step_tensor(step_size, dtype, device):
  """Scalar (or per-chain) step size as a device tensor of `dtype`."""
  if isinstance(step_size, (list, tuple)):
    vals = [torch.as_tensor(s) for s in step_size]
    first = vals[0]
    for v in vals[1:]:
      if not torch.equal(v.detach().cpu().double(), first.detach().cpu().double()):
        raise NotImplementedError(
            'per-part step sizes that differ are not built into the kernels')
    step_size = first
  # a Python number is filled in on the device: the copy of a pageable tensor
  # waits for the stream's earlier work
  if (type(step_size) is float and device.type == 'cuda' and
      abs(step_size) <= torch.finfo(dtype).max):
    return torch.full((1,), step_size, dtype=dtype, device=device)
  t = torch.as_tensor(step_size, dtype=dtype)
  return t.to(device).reshape(-1).contiguous()


class Run:
  """Owns the output buffers of one kernel launch."""

  def __init__(self, spec, table, state, tlp, grad, step, seed, n_iters=1,
               fold_seed=False, iter0=0, sampler='nuts'):
    _lib.require_cuda()
    self.spec = spec
    self.table = table
    self.state, self.tlp, self.grad = state, tlp, grad
    c, d = state.shape
    self.n_chains, self.dim = c, d
    self.step = step
    a = _lib.RunArgs()
    a.dtype = _lib.dtype_code(state.dtype)
    a.n_chains = c
    a.dim_stride = d
    a.max_dim = spec.dim
    a.n_iters = n_iters
    a.fold_seed = 1 if fold_seed else 0
    a.iter0 = int(iter0)
    seed = np.asarray(seed, np.uint32).reshape(2)
    a.seed[0], a.seed[1] = int(seed[0]), int(seed[1])
    a.target_kind = spec.kind
    if spec.kind in (_lib.TARGET_LOGISTIC, _lib.TARGET_LINEAR):
      base = getattr(spec, '_base', spec)
      # sampler: 'nuts' or 'hmc' (the HMC and MALA kernels)
      a.waves_per_chain = tuning.glm_waves(spec.kind, base.n_obs, base.dim,
                                           c, sampler, state.dtype)
    a.max_energy_diff = 1000.0
    a.problems = table.data_ptr()
    a.n_problems = 1
    a.step_size = step.data_ptr()
    if step.numel() == c and c > 1:
      self._chain_step = torch.arange(c, dtype=torch.int32, device=state.device)
      a.chain_step = self._chain_step.data_ptr()
    elif step.numel() != 1:
      raise ValueError(f'step size with {step.numel()} elements does not match '
                       f'{c} chains')
    a.state, a.tlp, a.grad = state.data_ptr(), tlp.data_ptr(), grad.data_ptr()
    self.args = a
    self.outputs = {}

  def want(self, name, shape, dtype):
    t = torch.empty(shape, dtype=dtype, device=self.state.device)
    self.outputs[name] = t
    setattr(self.args, name, t.data_ptr())
    return t

  def call_hmc(self, calibrated):
    """hipmc_hmc_run or hipmc_leapfrog_run, or the tiled trajectories where
    those are faster."""
    a = self.args
    if glm_tile.takes_trajectory(self.spec, a.max_dim, self.n_chains,
                                 a.num_leapfrog_steps):
      glm_tile.run_hmc(self.spec, a, calibrated, self.state.device)
      return self.outputs
    return self.call(_lib.lib().hipmc_hmc_run if calibrated
                     else _lib.lib().hipmc_leapfrog_run)

  def call(self, fn):
    _lib.check(fn(self.args, _lib.stream_handle(self.state.device)))
    return self.outputs


def flat_inputs(spec, parts, tlp, grads):
  """Packs state/grad parts; returns contiguous working copies."""
  # tlp has one element per chain in any shape: its own list
  state, grad, t = targets_lib.pack_states(
      [(parts, spec.event_shapes), (grads, spec.event_shapes),
       ([tlp], [()])], spec.dtype, spec.device)
  return state, t.reshape(-1), grad


def choose_lists(accepted, pairs):
  """choose_rows of several (proposed, current) pairs of lists, together where
  each pair's lists are as long as each other."""
  proposed, current = [], []
  for p, c in pairs:
    if len(p) != len(c):
      return [mcmc_util.choose(accepted, list(p), list(c)) for p, c in pairs]
    proposed += p
    current += c
  rows = choose_rows(accepted, proposed, current)
  out, at = [], 0
  for p, _ in pairs:
    out.append(rows[at:at + len(p)])
    at += len(p)
  return out


def choose_rows(accepted, proposed, current):
  """[torch.where(accepted, p, c)] of lists of per-chain tensors (as long as
  the shorter one), in one launch where they are equally many plain tensors of
  one type and shape on the current GPU."""
  n = accepted.numel()
  first = proposed[0]
  if (n == 0 or len(proposed) != len(current) or
      len(proposed) > _lib.MAX_COPY_BLOCKS or not first.is_cuda or
      first.device.index != torch.cuda.current_device() or
      first.element_size() not in (4, 8) or
      any(not isinstance(c, torch.Tensor) or c.requires_grad or
          c.is_neg() or p.is_neg() or
          c.dtype != first.dtype or p.dtype != first.dtype or
          c.device != first.device or c.shape != p.shape or
          p.shape[:accepted.dim()] != accepted.shape or
          not 0 < p.numel() < 1 << 31 for p, c in zip(proposed, current))):
    return mcmc_util.choose(accepted, list(proposed), list(current))
  out = [torch.empty(p.shape, dtype=p.dtype, device=p.device)
         for p in proposed]
  blocks = []
  for p, c, o in zip(proposed, current, out):
    p = p.reshape(n, -1)
    blocks.append((p, c.reshape(n, -1), o.data_ptr(), p.shape[1]))
  _lib.copy_blocks(blocks, first.element_size(), first.device, accepted)
  return out
