"""GPU test of zscore at lengths around its groups of 16 and its staged chunk
of 2048 entries, against the oracle; bar 1e-6 normwise, as the other zscore
test."""
import numpy as np
import pytest
import torch

from helpers import normwise_err
from tracetransform_amd import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 255, 360, 2047, 2048, 2049, 2064, 5001])
def test_zscore_lengths(oracle, gpu, n):
    x = (np.random.default_rng(n).random((3, n)) * 50 + 5).astype(np.float32)
    g = core.zscore(torch.from_numpy(x).cuda()).cpu().numpy()
    for k in range(3):
        assert normwise_err(g[k], oracle.zscore(x[k])) <= 1e-6
