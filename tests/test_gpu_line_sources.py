"""GPU tests of the two sources of the batched line kernels, pixel pairs and
the images with their row-major copies: the same bits as the single-image path
for every set of functionals the kernels are built for, forward and in the
backward's recompute, whichever is forced and whatever the rule chooses."""
import numpy as np
import pytest
import torch

from tracetransform_amd import _lib, core

pytestmark = pytest.mark.gpu


def images(sizes, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k, n in enumerate(sizes):
        x = rng.random((n, n), dtype=np.float32)
        if k % 3 == 1:
            x -= 0.4                      # negative samples
        if k % 3 == 2:                    # a zero border, huge and infinite pixels
            b = max(1, n // 6)
            x[:b] = x[-b:] = x[:, :b] = x[:, -b:] = 0.0
            x[n // 2, n // 2] = np.inf
            x[n // 2 - 1, n // 2] = 3e38
        out.append(torch.from_numpy(x).cuda())
    return out


def same(a, b):
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and torch.equal(
        torch.where(nan, 0, a.view(torch.int32)), torch.where(nan, 0, b.view(torch.int32)))


@pytest.mark.parametrize("codes", [[0], [1], [3], [0, 1, 2], [1, 3], [0, 1, 2, 3, 4, 5]])
def test_sources_give_the_same_bits(gpu, codes):
    L = _lib.load()
    imgs = images([3, 4, 5, 31, 32, 33, 64, 65, 70, 129, 130, 200], len(codes))
    A, step, pf = 24, 15.0, [(1,)]
    single = [core.sinograms(im, A, step, codes) for im in imgs]
    grads = []
    try:
        for pairs in (1, 0):
            L.tt_testing_line_pairs(pairs)
            for line in (None, (2, 32), (8, 16)):
                core.set_tiles(0, line=line)
                b = core.Batch(imgs, A, step, codes)
                b.run()
                for k in range(len(imgs)):
                    assert same(b.sino[k], single[k]), (pairs, line, k)
            core.set_tiles(0)
            finite = [im for k, im in enumerate(imgs) if k % 3 != 2]
            g = core.BatchBackward(finite, A, step, codes, pf)
            g.dcircus_all.fill_(0.25)
            grads.append([x.clone() for x in g.run()])
    finally:
        L.tt_testing_line_pairs(-1)
        core.set_tiles(0)
    assert all(same(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("A", [12, 13, 79, 80])
@pytest.mark.parametrize("codes", [[0], [0, 1, 3]])
def test_rule_on_a_large_batch(gpu, A, codes):
    # 510 images of 129 rows: more than 8 Mi pixels, the line between the
    # sources at 12.9 and, for T0 alone, at 80 angles
    base = images([129], 7)[0]
    imgs = [base * (1.0 + k / 510) for k in range(510)]
    b = core.Batch(imgs, A, 360.0 / A, codes)
    b.run()
    for k in (0, 255, 509):
        assert same(b.sino[k], core.sinograms(imgs[k], A, 360.0 / A, codes))
