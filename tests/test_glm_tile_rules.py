"""Which regressions' chains are tiled (host logic, no GPU): on each side of
the lines, and never past what the tiles hold."""

import types

import numpy as np
import pytest
import torch

from probability_amd import _lib
from probability_amd import glm_tile

F32, F64 = torch.float32, torch.float64
LOGISTIC, LINEAR = _lib.TARGET_LOGISTIC, _lib.TARGET_LINEAR


def _spec(kind, n, dtype):
  return types.SimpleNamespace(kind=kind, dtype=dtype,
                               base=types.SimpleNamespace(n_obs=n))


@pytest.mark.parametrize('dtype,kind,n,d,c,tiled', [
    (F32, LOGISTIC, 1199, 30, 64, False), (F32, LOGISTIC, 1200, 30, 1, True),
    (F32, LINEAR, 899, 64, 64, False), (F32, LINEAR, 900, 64, 64, True),
    (F32, LINEAR, 430, 256, 1, True), (F32, LINEAR, 429, 256, 1, False),
    (F32, LOGISTIC, 512, 2, 4095, False), (F32, LOGISTIC, 512, 2, 4096, True),
    (F32, LOGISTIC, 511, 2, 100000, False),
    (F32, LOGISTIC, 5000, 257, 64, False), (F32, LOGISTIC, 5000, 4, 0, False),
    (F64, LOGISTIC, 899, 30, 64, False), (F64, LOGISTIC, 900, 2, 64, True),
    (F64, LOGISTIC, 270, 100, 64, True), (F64, LOGISTIC, 269, 100, 64, False),
    (F64, LINEAR, 1399, 30, 64, False), (F64, LINEAR, 1400, 30, 64, True),
    (F64, LINEAR, 700, 100, 64, True), (F64, LINEAR, 5000, 129, 64, False)])
def test_evaluation(dtype, kind, n, d, c, tiled):
  dim = d + (kind == LINEAR)
  assert glm_tile.takes_eval(_spec(kind, n, dtype), dim, c) == tiled


@pytest.mark.parametrize('dtype,kind,n,d,c,leapfrogs,tiled', [
    (F32, LOGISTIC, 6001, 101, 512, 5, True),
    (F32, LOGISTIC, 3000, 30, 1, 10, True),
    (F32, LOGISTIC, 3000, 30, 1, 2, False),
    (F32, LOGISTIC, 2048, 8, 256, 10, False),  # two passes of four waves
    (F32, LOGISTIC, 512, 8, 2000, 10, False),
    (F32, LINEAR, 1024, 64, 512, 10, False),
    (F32, LINEAR, 2048, 64, 256, 10, False),
    (F32, LINEAR, 6000, 64, 64, 10, True),
    (F32, LOGISTIC, 700, 200, 1000, 3, True),
    (F64, LOGISTIC, 512, 64, 256, 10, False),
    (F64, LOGISTIC, 1024, 100, 64, 10, True),
    (F64, LOGISTIC, 512, 100, 256, 10, False),
    (F64, LINEAR, 2048, 30, 64, 10, False),
    (F64, LINEAR, 8000, 30, 64, 10, True),
    (F64, LINEAR, 8000, 129, 64, 10, False),
    (F32, LOGISTIC, 8000, 30, 64, 0, False)])
def test_trajectories(dtype, kind, n, d, c, leapfrogs, tiled):
  dim = d + (kind == LINEAR)
  assert glm_tile.takes_trajectory(_spec(kind, n, dtype), dim, c,
                                   leapfrogs) == tiled


@pytest.mark.parametrize('dtype,rows,cols,chains,tiled', [
    (F32, [600] * 16, 30, 16, False), (F32, [1300, 100], 30, 1, True),
    (F32, [600] * 256, 30, 16, True), (F32, [511] * 256, 30, 64, False),
    (F32, [2000] * 256, 30, 4, False), (F32, [2000] * 128, 30, 4, True),
    (F32, [600, 100], 200, 4, True), (F32, [2000], 257, 64, False),
    (F64, [2000] * 256, 4, 8, False), (F64, [2000] * 256, 17, 8, True),
    (F64, [2000] * 256, 4, 16, True), (F64, [2000], 129, 64, False)])
def test_batches(dtype, rows, cols, chains, tiled):
  n = len(rows)
  tiles = glm_tile.BatchTiles(rows, cols, [chains] * n,
                              np.arange(n + 1) * chains, dtype, 'cpu')
  assert (tiles.table is not None) == tiled
  if tiled:
    t = tiles.table.numpy()
    per = t[:, 5]
    assert t[:, 2].sum() == n * chains and (per % 64 == 0).all()
    assert (t[:, 3] * per >= np.asarray(rows)[t[:, 0]]).all()
    assert tiles.slots == t[:, 3].sum() and tiles.max_split == t[:, 3].max()
