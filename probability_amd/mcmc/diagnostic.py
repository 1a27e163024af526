"""ESS and potential scale reduction on the device
(`mcmc/diagnostic.py:38-568`, `stats/sample_stats.py:44-216`).

Same formulas as the reference: centred FFT auto-covariance zero-padded to
2^ceil(log2(2n)) divided by (n - k); cross-chain ESS (Vehtari et al. 2021
eq. 10) truncated at the first negative auto-correlation; split R-hat.
Computed in float64: float32 and float64 draws on the GPU by libhipmc
(csrc/diagnostic.hip: the cross-chain ESS of up to 4096 draws, and R-hat),
everything else with torch.
"""

import math

import numpy as np
import torch

from probability_amd import _lib

__all__ = ['effective_sample_size', 'potential_scale_reduction']


def _as64(x):
  if isinstance(x, torch.Tensor):
    return x.to(torch.float64)
  return torch.as_tensor(x, dtype=torch.float64)


# The most draws whose zero-padded transform fits in one workgroup's LDS.
_MAX_DRAWS = 4096


def _on_device(x):
  """Whether the kernels take x: a plain float tensor on the GPU that no
  transformation (autograd, forward mode, vmap, tracing) follows."""
  return (type(x) is torch.Tensor and x.is_cuda and
          x.dtype in (torch.float32, torch.float64) and
          not (x.requires_grad and torch.is_grad_enabled()) and
          torch.autograd.forward_ad._current_level < 0 and
          not torch._C._functorch.is_functorch_wrapped_tensor(x) and
          not torch.compiler.is_compiling())


def _ess_takes(n, c, d):
  """Whether the ESS of n draws of c chains of d dimensions is the kernels':
  within their limits (a grid holds fewer than 2^32 threads), and not where the
  torch form is faster: few draws, since a block's fixed work per pair of chains
  is that of 64 threads, and short series of very many chains, which few blocks
  share.  us, torch form / kernels: 4 draws, 25000 x 3 series 241 / 252, 2 x
  1000000 1012 / 1665; 8 draws, 2000 x 500 1113 / 1131, 100000 x 1 275 / 690; 17
  draws, 20000 x 50 4248 / 1344, 250000 x 1 1383 / 1684; 65 draws, 250000 x 1
  7130 / 1812."""
  if not (n <= _MAX_DRAWS and 2 <= c <= 1 << 30 and c * d < 1 << 30 and
          d * max(64, n // 4) < 1 << 32):
    return False
  return n > 64 or c * d <= 50000 or (n > 8 and c <= 65536)


def _rhat_takes(x, chain_axes):
  """Whether R-hat of draws x [n, chain axes..., ...] is the kernels': within
  their limits, and not for few draws of very many series, where a pass over
  memory takes less than the kernels' fixed work per series.  Split R-hat, us,
  torch form / kernels: 8 draws of 600000 series 69 / 77, of 2000000 152 / 228;
  float64, 34 draws of 1200000 185 / 203; 48 draws of 1200000 series 440 / 207,
  65 draws of 2000000 881 / 230."""
  n, series = x.shape[0], math.prod(x.shape[1:])
  if not (isinstance(chain_axes, int) and chain_axes < x.dim() and
          0 < series < 1 << 30 and n <= 1 << 30 and
          math.prod(x.shape[1:1 + chain_axes]) <= 1 << 29):
    return False
  return n > 40 or series < 500000


def _series(x, chain_axes):
  """x [n, chain axes..., rest...] as [n, chains, dims] (a view where the
  strides allow)."""
  chains = math.prod(x.shape[1:1 + chain_axes])
  return x.reshape(x.shape[0], chains, math.prod(x.shape[1 + chain_axes:]))


def _ess_device(states, filter_threshold):
  """states [n, chains, ...] -> cross-chain ESS [...]."""
  x = _series(states, 1)
  n, c, d = x.shape
  # blocks that share a dimension's pairs of chains: two blocks a CU are
  # resident, so up to 512 run at once; none is empty
  pairs = (c + 1) // 2
  per = -(-pairs // min(pairs, max(1, 512 // d)))
  blocks = -(-pairs // per)
  m = max(16, 1 << (2 * n - 1).bit_length())
  f64 = dict(dtype=torch.float64, device=x.device)
  rows = torch.empty((d, c, n), dtype=x.dtype, device=x.device)
  means = torch.empty((d, c), **f64)
  power = torch.empty((blocks, d, m), **f64)
  out = torch.empty(d, **f64)
  with torch.cuda.device(x.device):
    _lib.check(_lib.lib().hipmc_effective_sample_size(
        _lib.dtype_code(x.dtype), n, c, d, *x.stride(), _lib.ptr(x),
        0 if filter_threshold is None else 1,
        0.0 if filter_threshold is None else float(filter_threshold), blocks,
        _lib.ptr(rows), _lib.ptr(means), _lib.ptr(power), _lib.ptr(out),
        _lib.stream_handle(x.device)))
  return out.reshape(states.shape[2:])


def _rhat_device(state, independent_chain_ndims, split_chains):
  """state [n, chain axes..., ...] -> R-hat [...]."""
  x = _series(state, independent_chain_ndims)
  n, c, d = x.shape
  halves = 2 if split_chains else 1
  # a block takes up to 64 adjacent series, its other threads 16 draws at a
  # time; time chunks so that about 2048 blocks run, none with less than one
  # such step, and so many that merging them (0.2 us each, in a row) takes as
  # long as the steps of one (1.5 us each)
  width = min(64, 1 << (c * d - 1).bit_length())
  blocks = halves * -(-(c * d) // width)
  steps = -(-(n // halves) // (16 * (256 // width)))
  chunks = max(1, min(2048 // blocks, steps, math.isqrt(8 * steps)))
  sums = torch.empty((chunks, halves, 2, c * d), dtype=torch.float64,
                     device=x.device)
  out = torch.empty(d, dtype=torch.float64, device=x.device)
  with torch.cuda.device(x.device):
    _lib.check(_lib.lib().hipmc_potential_scale_reduction(
        _lib.dtype_code(x.dtype), n, c, d, *x.stride(), _lib.ptr(x),
        1 if split_chains else 0, chunks, _lib.ptr(sums), _lib.ptr(out),
        _lib.stream_handle(x.device)))
  return out.reshape(state.shape[1 + independent_chain_ndims:])


def auto_covariance(x):
  """x [n, ...] -> auto-covariance along axis 0 (unnormalised)."""
  x = _as64(x)
  n = x.shape[0]
  x = x - x.mean(0, keepdim=True)
  m = int(2 ** math.ceil(math.log2(2 * n)))
  f = torch.fft.rfft(x, n=m, dim=0)
  ac = torch.fft.irfft(f * f.conj(), n=m, dim=0)[:n]
  k = torch.arange(n, dtype=torch.float64, device=x.device)
  return ac / (n - k).reshape((-1,) + (1,) * (x.dim() - 1))


def _flatten_chain_dims(states, cross_chain_dims):
  """Moves the chain dimensions (an int or a sequence of ints, counted in
  `states`) to axis 1 as one flattened chain axis."""
  dims = ([cross_chain_dims] if isinstance(cross_chain_dims, int)
          else [int(d) for d in cross_chain_dims])
  dims = [d % states.dim() for d in dims]
  if 0 in dims:
    raise ValueError('cross_chain_dims cannot include the sample axis 0')
  rest = [d for d in range(1, states.dim()) if d not in dims]
  x = states.permute([0] + dims + rest)
  return x.reshape((x.shape[0], -1) + tuple(states.shape[d] for d in rest))


def _ess_one(states, cross_chain_dims, filter_threshold):
  # the kernel takes one threshold for all dimensions; a tensor that
  # broadcasts over them (or lies on the GPU) goes to the torch form
  number = filter_threshold is None or isinstance(
      filter_threshold, (int, float, np.integer, np.floating))
  if (cross_chain_dims is not None and number and _on_device(states) and
      states.dim() > 1):
    x = _flatten_chain_dims(states, cross_chain_dims)
    if x.numel() > 0 and _ess_takes(*x.shape[:2], math.prod(x.shape[2:])):
      return _ess_device(x, filter_threshold)
  states = _as64(states)
  if cross_chain_dims is not None:
    states = _flatten_chain_dims(states, cross_chain_dims)
  n = states.shape[0]
  ac = auto_covariance(states)
  if cross_chain_dims is not None:
    c = states.shape[1]
    if c < 2:
      raise ValueError('When `cross_chain_dims` is not `None`, there must be '
                       '> 1 chain in `states`.')
    b_div_n = states.mean(0).var(dim=0, unbiased=True)
    w = ac[0].mean(0)
    approx = w + b_div_n
    rho = 1.0 - (w - ac.mean(1)) / approx
  else:
    c = 1
    rho = ac / ac[:1]
  k = torch.arange(rho.shape[0], dtype=torch.float64, device=rho.device)
  nk = ((n - k) / n).reshape((-1,) + (1,) * (rho.dim() - 1))
  wr = nk * rho
  if filter_threshold is not None:
    mask = (rho < filter_threshold).to(torch.float64)
    mask = torch.clamp(1.0 - torch.cumsum(mask, 0), min=0.0)
    wr = wr * mask
  return c * n / (-1.0 + 2.0 * wr.sum(0))


def effective_sample_size(states, filter_threshold=0., filter_beyond_lag=None,
                          filter_beyond_positive_pairs=False,
                          cross_chain_dims=None, validate_args=False,
                          name=None):
  """ESS of each state part ([n, chains, ...] -> [...])."""
  if filter_beyond_lag is not None or filter_beyond_positive_pairs:
    raise NotImplementedError('only the default truncation rule is built')
  if isinstance(states, (list, tuple)):
    cdims = (cross_chain_dims if isinstance(cross_chain_dims, (list, tuple))
             else [cross_chain_dims] * len(states))
    return [_ess_one(s, cd, filter_threshold) for s, cd in zip(states, cdims)]
  return _ess_one(states, cross_chain_dims, filter_threshold)


def _rhat_one(state, independent_chain_ndims, split_chains):
  x = state if _on_device(state) else _as64(state)
  icn = independent_chain_ndims
  if icn < 1:
    raise ValueError('Argument `independent_chain_ndims` must be `>= 1`, '
                     'found: {}'.format(icn))
  if not split_chains and x.shape[0] < 2:
    raise ValueError('Must provide at least 2 samples. Found {}'.format(
        x.shape[0]))
  if split_chains:
    n = x.shape[0]
    if n < 4:
      raise ValueError('Must provide at least 4 samples when splitting '
                       'chains. Found {}'.format(n))
  if _on_device(x):
    if _rhat_takes(x, icn):
      return _rhat_device(x, icn, split_chains)
    x = _as64(x)
  if split_chains:
    n = x.shape[0]
    x = x[:n - n % 2]
    x = x.reshape((2, n // 2) + tuple(x.shape[1:])).transpose(0, 1)
    icn += 1
  n = x.shape[0]
  chain_axes = tuple(range(1, 1 + icn))
  all_axes = tuple(range(0, 1 + icn))
  m = 1
  for a in chain_axes:
    m *= x.shape[a]
  means = x.mean(0, keepdim=True)
  b_div_n = means.var(dim=all_axes, unbiased=True)
  w = x.var(dim=0, unbiased=True, keepdim=True).mean(dim=all_axes)
  s2 = ((n - 1) / n) * w + b_div_n
  return ((m + 1.0) / m) * s2 / w - (n - 1.0) / (m * n)


def potential_scale_reduction(chains_states, independent_chain_ndims=1,
                              split_chains=False, validate_args=False,
                              name=None):
  """R-hat of each state part ([n, chains, ...] -> [...])."""
  if isinstance(chains_states, (list, tuple)):
    return [_rhat_one(s, independent_chain_ndims, split_chains)
            for s in chains_states]
  return _rhat_one(chains_states, independent_chain_ndims, split_chains)
