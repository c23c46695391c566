"""GPU test of the transposed rotation at the edges of its pixel tiles (30 x 32
pixels, tiles that hang over the image, images smaller than a tile) and of its
item numbering (classes of one, two and three passes over the angles), against
the oracle's FP64 vector-Jacobian product; bar 1e-5 normwise, as the other
adjoint tests."""
import numpy as np
import pytest
import torch

from helpers import normwise_err
from tracetransform_amd import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("codes", [[0], [0, 2], [0, 3, 4, 5], [0, 1, 2, 3, 4, 5]])
@pytest.mark.parametrize("n", [3, 5, 29, 30, 31, 32, 33, 34, 61, 64, 65, 91, 129])
def test_image_gradient_at_tile_edges(oracle, gpu, n, codes):
    A, step = 77, 360.0 / 76  # 0 and 90 degrees among them, others irregular
    rng = np.random.default_rng(100 * n + len(codes))
    img = (rng.random((n, n)) + 0.05).astype(np.float32)
    _, aux = oracle.sinograms(img.ravel(), n, A, step, codes, nthreads=8)
    ds = rng.standard_normal((len(codes), A, n)).astype(np.float32)
    got = core.sinograms_backward(torch.from_numpy(img).cuda(), A, step, codes,
                                  torch.from_numpy(ds).cuda())
    want = oracle.sinograms_vjp_f64(img.ravel(), n, A, step, codes, aux, ds, nthreads=8)
    assert normwise_err(got.cpu().numpy().ravel(), want) <= 1e-5
