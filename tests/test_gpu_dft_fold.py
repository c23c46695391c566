"""GPU tests of P3's folded DFT products and their adjoint at the edges of
their tiles (64 or 128 rows and columns, chunks of 16 of the folded reduction)
and of the fold (odd and even lengths, the shortest columns), against numpy's
FP64 transform; normwise bar 1e-5, as the other value tests."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import normwise_err
from tracetransform_amd import _lib, core

pytestmark = pytest.mark.gpu


def trapz_weights(n):
    lin = (-1 + np.arange(n) * 2.0 / (n - 1)).astype(np.float32).astype(np.float64)
    w = np.zeros(n)
    w[1:] += 0.5 * np.diff(lin)
    w[:-1] += 0.5 * np.diff(lin)
    return w


@pytest.mark.parametrize("n", [3, 4, 5, 8, 30, 31, 32, 33, 63, 64, 126, 127, 128, 129, 255, 258,
                               363])
@pytest.mark.parametrize("cols", [1, 65, 130])
def test_p3_and_adjoint(gpu, n, cols):
    rng = np.random.default_rng(1000 * n + cols)
    x = (rng.random((2, cols, n)) + 0.1 * rng.standard_normal((2, cols, n))).astype(np.float32)
    dc = rng.standard_normal((2, 1, cols)).astype(np.float32)
    xt = torch.from_numpy(x).cuda()
    got = core.circus(xt, [(3,)])[:, 0].cpu().numpy()
    grad = core.circus_backward(xt, [(3,)], torch.from_numpy(dc).cuda()).cpu().numpy()
    w = trapz_weights(n)
    f = np.fft.fft(x.astype(np.float64), axis=-1)
    m = np.abs(f) ** 2
    want = (w * m * m).sum(-1) / float(n) ** 4
    dwant = 4.0 / float(n) ** 4 * np.fft.fft(w * m * np.conj(f), axis=-1).real
    dwant *= dc[:, 0, :, None].astype(np.float64)
    assert normwise_err(got, want) <= 1e-5
    assert normwise_err(grad, dwant) <= 1e-5


# columns that just do not fill the last tile: 64 x 128 tiles (also where 128
# rows would be half empty), 128 x 128 tiles, both directions
@pytest.mark.parametrize("n,cols,forward,adjoint", [
    (3, 33001, (64, 128), (64, 128)), (62, 17001, (64, 128), (64, 128)),
    (63, 70003, (64, 128), (64, 128)), (126, 70003, (64, 128), (64, 128)),
    (129, 11017, (64, 128), (64, 128)), (362, 9001, (64, 128), (64, 128)),
    (129, 66049, (128, 128), (128, 128)), (255, 65573, (128, 128), (128, 128)),
    (362, 33001, (128, 128), (128, 128))])
def test_wide_tiles(gpu, n, cols, forward, adjoint):
    for fwd, shape in ((1, forward), (0, adjoint)):
        bm, bn = C.c_int(), C.c_int()
        assert _lib.load().tt_testing_dft_shape(n, cols, fwd, C.byref(bm), C.byref(bn)) == 0
        assert (bm.value, bn.value) == shape, fwd
    rng = np.random.default_rng(n + cols)
    x = (rng.random((cols, n)) + 0.1 * rng.standard_normal((cols, n))).astype(np.float32)
    dc = rng.standard_normal((1, 1, cols)).astype(np.float32)
    xt = torch.from_numpy(x[None]).cuda()
    got = core.circus(xt, [(3,)])[0, 0].cpu().numpy()
    grad = core.circus_backward(xt, [(3,)], torch.from_numpy(dc).cuda())[0].cpu().numpy()
    w = trapz_weights(n)
    f = np.fft.fft(x.astype(np.float64), axis=-1)
    m = np.abs(f) ** 2
    want = (w * m * m).sum(-1) / float(n) ** 4
    dwant = 4.0 / float(n) ** 4 * np.fft.fft(w * m * np.conj(f), axis=-1).real
    dwant *= dc[0, 0, :, None].astype(np.float64)
    assert normwise_err(got, want) <= 1e-5
    assert normwise_err(grad, dwant) <= 1e-5
