"""GPU tests of the line kernels and the transposed rotation at the largest
sides they take (2730 and 1800 rows): medians and T0 bit for bit, T1..T5 and
gradients within 1e-5 of FP64, both line sources of a batch the single-image
path's bits."""
import numpy as np
import pytest
import torch

from helpers import assert_same_indices, normwise_err
from tracetransform_amd import _lib, core

pytestmark = pytest.mark.gpu


def image(kind, n, seed):
    img = np.random.default_rng(seed).random((n, n), dtype=np.float32)
    if kind == "inner":
        b = n // 6
        out = np.zeros_like(img)
        out[b:-b, b:-b] = img[b:-b, b:-b]
        return out
    return img + np.float32(0.25) if kind == "full" else img - np.float32(0.3)


@pytest.mark.parametrize("n,kind", [(1450, "full"), (2000, "full"), (2000, "signed"),
                                    (2729, "inner"), (2730, "full"), (2730, "signed")])
def test_line_kernel(oracle, gpu, n, kind):
    A, step, codes = 8, 37.0, [0, 1, 2, 3, 4, 5]
    img = image(kind, n, n)
    sino, aux = core.sinograms(torch.from_numpy(img).cuda(), A, step, codes, with_aux=True)
    g = sino.cpu().numpy()
    o, oaux = oracle.sinograms(img.ravel(), n, A, step, codes, nthreads=8)
    assert_same_indices("median_x", aux["median_x"].cpu(), oaux["med_x"])
    assert_same_indices("median_sqrt", aux["median_sqrt"].cpu(), oaux["med_s"])
    assert np.array_equal(g[0], o[0])
    d = oracle.sinograms_f64(img.ravel(), n, A, step, codes, oaux, nthreads=8, geometry=1)
    for t in range(1, 6):
        assert normwise_err(g[t], d[t]) <= 1e-5, t


@pytest.mark.parametrize("codes", [[0], [0, 1, 2, 3, 4, 5]])
def test_batch_sources(gpu, codes):
    imgs = [torch.from_numpy(image(k, n, n)).cuda()
            for n, k in ((2730, "full"), (2729, "signed"), (2000, "inner"), (1451, "full"))]
    A, step = 9, 37.0
    single = [core.sinograms(im, A, step, codes) for im in imgs]
    try:
        for pairs in (1, 0):
            _lib.load().tt_testing_line_pairs(pairs)
            b = core.Batch(imgs, A, step, codes)
            b.run()
            for k in range(len(imgs)):
                assert torch.equal(b.sino[k], single[k]), (pairs, k)
    finally:
        _lib.load().tt_testing_line_pairs(-1)


@pytest.mark.parametrize("n,codes", [(1450, [0, 3]), (1799, [0]), (1800, [0, 1, 2, 3, 4, 5])])
def test_gradient(oracle, gpu, n, codes):
    A, step = 7, 51.0
    img = image("full", n, n)
    _, aux = oracle.sinograms(img.ravel(), n, A, step, codes, nthreads=8)
    ds = np.random.default_rng(n).standard_normal((len(codes), A, n)).astype(np.float32)
    got = core.sinograms_backward(torch.from_numpy(img).cuda(), A, step, codes,
                                  torch.from_numpy(ds).cuda())
    want = oracle.sinograms_vjp_f64(img.ravel(), n, A, step, codes, aux, ds, nthreads=8)
    assert normwise_err(got.cpu().numpy().ravel(), want) <= 1e-5
