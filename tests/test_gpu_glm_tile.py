"""The tiled GLM evaluation (many chains' logits and gradients as matrix
products) at the edges of its tiles: rows off the 16-row sub-tiles and 64-row
passes, columns off the 16-column slabs, chains off the 16- and 32-chain
tiles, both types and models, bijectors on every part.

Densities, gradients and trajectories are held to the float64 oracle at the
parity bar of the per-chain kernels: 1e-5 normwise in float32, 1e-11 in
float64.  Whole runs (accepts, traces, per-chain steps, momentum precision)
are compared with the per-chain kernel: the same decisions, states to the
same bounds."""

import numpy as np
import pytest
import torch

from oracle import mcmc as omcmc
from oracle import rng as orng
from oracle import targets as otg
from probability_amd import _lib
from probability_amd import bijectors as pbij
from probability_amd import glm_tile
from probability_amd import targets as ptg
from probability_amd.mcmc import _runner
from probability_amd.mcmc import batched

pytestmark = pytest.mark.gpu

TYPES = [(torch.float32, np.float32, 1e-5), (torch.float64, np.float64, 1e-11)]


def _normwise(got, want, tol):
  got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
  assert got.shape == want.shape
  assert np.abs(got - want).max() <= tol * max(np.abs(want).max(), 1.0)


def _case(model, n, d, c, ndt, seed, beta_code=0):
  """(spec, oracle target, chains)."""
  r = np.random.default_rng(seed)
  tdt = torch.float32 if ndt == np.float32 else torch.float64
  x = r.normal(size=(n, d)).astype(ndt)
  b = r.normal(size=d) / np.sqrt(d)
  s = x.astype(np.float64) @ b
  bij = [pbij.Identity(), pbij.Softplus(), pbij.Exp()][beta_code]
  if model == 'logistic':
    y = (r.uniform(size=n) < 1 / (1 + np.exp(-s))).astype(ndt)
    spec = ptg.LogisticRegression(x, y, prior_scale=1.5, dtype=tdt)
    o = otg.LogisticRegression(x.astype(np.float64), y.astype(np.float64),
                               prior_scale=1.5)
    codes = np.full(d, beta_code, np.int32)
    if beta_code:
      spec = ptg.TransformedTarget(spec, [bij])
  else:
    y = (s + 0.7 * r.normal(size=n)).astype(ndt)
    spec = ptg.TransformedTarget(
        ptg.LinearRegression(x, y, sigma_scale=2.0, dtype=tdt),
        [bij, pbij.Exp()])
    o = otg.LinearRegression(x.astype(np.float64), y.astype(np.float64),
                             sigma_scale=2.0)
    codes = np.concatenate([np.full(d, beta_code, np.int32), [2]])
  q = np.concatenate([b + 0.1 * r.normal(size=(c, d)),
                      np.log(0.7) + 0.05 * r.normal(size=(c, 1))], 1)
  q = q[:, :spec.dim].astype(ndt)
  ot = otg.Transformed(o, codes) if codes.any() else o
  return spec, ot, q


def _evaluate(spec, q):
  x = torch.as_tensor(q, device='cuda')
  tlp, grad = torch.empty_like(x[:, 0]), torch.empty_like(x)
  table = spec.table(spec.bijectors_for_eval())
  glm_tile.evaluate(spec, table, x, tlp, grad)
  return tlp.cpu().numpy(), grad.cpu().numpy()


SHAPES = [(1, 1, 1), (15, 3, 16), (16, 16, 17), (17, 17, 15), (63, 31, 33),
          (64, 32, 32), (65, 33, 31), (129, 64, 50), (512, 65, 7),
          (513, 100, 64), (1000, 112, 100), (640, 127, 65), (700, 128, 20)]


@pytest.mark.parametrize('tdt,ndt,tol', TYPES)
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('n,d,c', SHAPES)
def test_density_and_gradient_match_oracle(n, d, c, model, tdt, ndt, tol):
  spec, o, q = _case(model, n, d, c, ndt, n + d + c)
  t, g = o.log_prob_and_grad(q.astype(np.float64))
  tlp, grad = _evaluate(spec, q)
  _normwise(tlp, t, tol)
  _normwise(grad, g, tol)


@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('n,d,c', [(600, 129, 40), (333, 200, 16),
                                   (530, 255, 3), (90, 256, 18)])
def test_wide_float32_designs_match_oracle(n, d, c, model):
  spec, o, q = _case(model, n, d, c, np.float32, d)
  t, g = o.log_prob_and_grad(q.astype(np.float64))
  tlp, grad = _evaluate(spec, q)
  _normwise(tlp, t, 1e-5)
  _normwise(grad, g, 1e-5)


@pytest.mark.parametrize('tdt,ndt,tol', TYPES)
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('code', [1, 2])
def test_bijectors_on_the_coefficients_match_oracle(code, model, tdt, ndt, tol):
  spec, o, q = _case(model, 200, 21, 37, ndt, 5, beta_code=code)
  t, g = o.log_prob_and_grad(q.astype(np.float64))
  tlp, grad = _evaluate(spec, q)
  _normwise(tlp, t, tol)
  _normwise(grad, g, tol)


def _leapfrog(spec, q, eps, steps, seed):
  x = torch.as_tensor(q, device='cuda').clone()
  tlp, grad = spec.log_prob_and_grad_flat(x)
  step = torch.full((1,), float(eps), dtype=x.dtype, device='cuda')
  run = _runner.Run(spec, spec.table(spec.bijectors_for_eval()), x, tlp, grad,
                    step, seed, sampler='hmc')
  run.args.num_leapfrog_steps = steps
  p0 = run.want('out_initial_momentum', x.shape, x.dtype)
  p1 = run.want('out_final_momentum', x.shape, x.dtype)
  corr = run.want('out_energy', (1, x.shape[0]), x.dtype)
  glm_tile.run_hmc(spec, run.args, False, x.device)
  return [v.cpu().numpy() for v in (x, tlp, grad, p0, p1, corr[0])]


@pytest.mark.parametrize('tdt,ndt,tol', TYPES)
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('n,d,c,steps', [(65, 5, 3, 1), (200, 33, 16, 2),
                                         (1300, 64, 33, 4), (520, 100, 70, 3)])
def test_trajectories_match_oracle(n, d, c, steps, model, tdt, ndt, tol):
  spec, o, q = _case(model, n, d, c, ndt, n)
  eps, seed = ndt(0.01), orng.sanitize_seed(n)
  x, t, g, p0, p1, corr = _leapfrog(spec, q, eps, steps, seed)
  qd = q.astype(np.float64)
  t0, g0 = o.log_prob_and_grad(qd)
  want0 = orng.PhiloxDraws(ndt).momentum(seed, c, spec.dim).astype(np.float64)
  w1, wq, wt, wg = omcmc.leapfrog(o, float(eps), steps, want0, qd, t0, g0)
  _normwise(p0, want0, tol)
  _normwise(x, wq, tol)
  _normwise(t, wt, tol)
  _normwise(g, wg, tol)
  _normwise(p1, w1, tol)
  # a difference of kinetic energies, bounded relative to them
  ke = 0.5 * (want0 ** 2).sum(1).max()
  assert np.abs(corr - 0.5 * ((want0 ** 2).sum(1) - (w1 ** 2).sum(1))).max() \
      <= 10 * tol * max(ke, 1.0)


@pytest.mark.parametrize('tdt,ndt,tol', TYPES)
@pytest.mark.parametrize('model', ['logistic', 'linear'])
@pytest.mark.parametrize('precision', [False, True])
def test_runs_equal_the_per_chain_kernel(precision, model, tdt, ndt, tol):
  """Five calibrated transitions with per-chain steps, a thinned trace and
  every output, from the same start."""
  n, d, c, iters = 300, 40, 37, 5
  spec, _, q = _case(model, n, d, c, ndt, 11)
  dev, dim = 'cuda', spec.dim
  r = np.random.default_rng(0)
  steps = torch.as_tensor((0.01 * r.uniform(0.5, 1.5, c)).astype(ndt),
                          device=dev)
  prec = torch.as_tensor(r.uniform(0.5, 2.0, (1, dim)).astype(ndt), device=dev)
  outs = []
  for tiled in (False, True):
    x = torch.as_tensor(q, device=dev).clone()
    tlp, grad = spec.log_prob_and_grad_chains(x)
    run = _runner.Run(spec, spec.table(spec.bijectors_for_eval()), x, tlp,
                      grad, steps, [3, 4], n_iters=iters, fold_seed=True,
                      iter0=2, sampler='hmc')
    a = run.args
    a.num_leapfrog_steps, a.out_row0 = 4, 1
    if precision:
      a.momentum_precision = prec.data_ptr()
    shapes = dict(out_log_accept_ratio=(iters + 1, c),
                  out_energy=(iters + 1, c),
                  out_target_log_prob=(iters + 1, c),
                  out_proposed_state=(c, dim), out_proposed_tlp=(c,),
                  out_initial_momentum=(c, dim), out_final_momentum=(c, dim),
                  trace_state=(2, c, dim))
    got = {k: run.want(k, s, tdt).zero_() for k, s in shapes.items()}
    acc = run.want('out_is_accepted', (iters + 1, c), torch.uint8).zero_()
    a.trace_start, a.trace_every, a.n_trace = 3, 2, 2
    if tiled:
      glm_tile.run_hmc(spec, a, True, x.device)
    else:
      run.call(_lib.lib().hipmc_hmc_run)
    got.update(state=x, tlp=tlp, grad=grad)
    outs.append(({k: v.cpu().numpy() for k, v in got.items()},
                 acc.cpu().numpy()))
  (want, wa), (got, ga) = outs
  np.testing.assert_array_equal(ga, wa)
  for k in want:
    # ratios of densities are bounded by the densities themselves
    scale = (np.abs(want['tlp']).max() if k in (
        'out_log_accept_ratio', 'out_energy') else 1.0)
    assert np.abs(got[k].astype(np.float64) - want[k]).max() <= \
        10 * tol * max(np.abs(want[k]).max(), scale), k


@pytest.mark.parametrize('tdt,ndt,tol', TYPES)
@pytest.mark.parametrize('chains', [[5, 16, 1, 9], [32, 50, 33, 7]])
def test_batch_of_ragged_regressions_matches_oracle(chains, tdt, ndt, tol):
  cases = [_case('logistic', 130, 7, chains[0], ndt, 1),
           _case('linear', 2100, 60, chains[1], ndt, 2),
           _case('logistic', 64, 33, chains[2], ndt, 3),
           _case('linear', 17, 1, chains[3], ndt, 4, beta_code=1)]
  batch = batched.PosteriorBatch(
      [s.base for s, _, _ in cases], chains,
      bijectors=[s.bijectors for s, _, _ in cases], slot_dim=70)
  x = torch.zeros((batch.n_chains, batch.dim_stride), dtype=tdt, device='cuda')
  for q, view in zip((q for _, _, q in cases), batch.split(x)):
    view.copy_(torch.as_tensor(q))
  tlp, grad = batch.eval(x)
  assert batch._tiles.table is not None
  ends = np.cumsum([0] + chains)
  for i, (_, o, q) in enumerate(cases):
    t, g = o.log_prob_and_grad(q.astype(np.float64))
    _normwise(tlp[ends[i]:ends[i + 1]].cpu().numpy(), t, tol)
    _normwise(batch.split(grad)[i].cpu().numpy(), g, tol)
  for i, d in enumerate(batch.dims):
    assert not bool(grad[ends[i]:ends[i + 1], d:].any())
