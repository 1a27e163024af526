"""ESS of dimensions whose pairs of chains go through one block in a row: the
next pair's loads during a transform, the transform's buffer used again, the
power added over the pairs, in blocks of one to sixteen waves.  Tolerances as
over the sizes."""

import numpy as np
import pytest
import torch

import test_gpu_diagnostic_sizes as sizes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,c,d', [
    (70, 12, 500), (200, 17, 129), (300, 7, 260), (600, 21, 130),
    (1000, 33, 127), (2100, 9, 300), (4096, 8, 257)])
@pytest.mark.parametrize('dtype', [np.float32, np.float64])
def test_blocks_of_several_pairs_match_oracle(n, c, d, dtype):
  pairs = (c + 1) // 2
  assert -(-pairs // min(pairs, max(1, 512 // d))) >= 3
  x = sizes._draws(n, c, d, dtype, n + c + d)
  sizes._check(x, torch.as_tensor(x, device='cuda'))
