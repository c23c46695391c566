"""GPU tests of the batched paths' pixel-pair workspace: bounded for large
batches, smaller where the device has no room for it, and the results the same
bits whatever share of the batch it holds at a time."""
import ctypes as C

import numpy as np
import pytest
import torch

from tracetransform_amd import _lib, core

pytestmark = pytest.mark.gpu


def test_pair_workspace_in_groups(gpu, monkeypatch):
    # where the device has no room for the pixel pairs of the whole batch,
    # groups of its images share a smaller workspace: the same bits, tuned or
    # not, and out of memory only where one image's pairs do not fit
    L = _lib.load()
    rng = np.random.default_rng(3)
    imgs = [torch.from_numpy(rng.random((n, n), dtype=np.float32)).cuda()
            for n in [97, 129, 33, 129, 120, 64, 97] * 2]
    codes, pf, A = [0, 1, 3], [(1,), (3,)], 8
    pairs = 2 * 8 * sum(im.numel() for im in imgs)
    largest = 2 * 8 * (129 * 129 + 2)
    limit = 2 * largest + 1000
    assert 3 * limit < pairs

    def run(limit, autotune=False):
        monkeypatch.setattr(core._tls, "ctx", {}, raising=False)  # no workspaces yet
        L.tt_testing_limit_allocation(C.c_size_t(limit))
        try:
            fwd = core.Batch(imgs, A, 45.0, codes, pf, save_for_backward=True)
            bwd = core.BatchBackward(imgs, A, 45.0, codes, pf)
            bwd.dcircus_all.fill_(0.25)
            out = []
            for _ in range(2):  # planned, then replayed
                sino, circ = fwd.run(autotune=autotune)
                out += [x.clone() for x in sino + circ + bwd.run()]
            torch.cuda.synchronize()
            return out
        finally:
            L.tt_testing_limit_allocation(C.c_size_t(0))

    ref = run(0)
    for got in (run(limit), run(limit, autotune=True)):
        assert all(torch.equal(a, b) for a, b in zip(ref, got))
    with pytest.raises(_lib.TTError, match="out of memory"):
        run(largest - 100)


def test_pair_workspace_of_a_large_batch(gpu, monkeypatch):
    # the pairs take 16 bytes a pixel, four times the images: bounded, however
    # large the batch
    monkeypatch.setattr(core._tls, "ctx", {}, raising=False)
    n, count, A = 1449, 300, 4
    img = torch.rand((n, n), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    imgs = [img * (1.0 + k / count) for k in range(count)]
    b = core.Batch(imgs, A, 90.0, [0, 1])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    b.run()
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    print(f"[pairs] {16 * n * n * count / 2**30:.2f} GiB of pairs, {used / 2**30:.2f} GiB used")
    assert 16 * n * n * count > 9 * 2**30 and used < 8.6 * 2**30
    for k in (0, count // 2, count - 1):
        assert torch.equal(b.sino[k], core.sinograms(imgs[k], A, 90.0, [0, 1]))
