"""GPU tests of the T0..T5 line kernel's schedule and square root.

* The line kernel's root (v_rsq_f32 and one Newton step) equals the correctly
  rounded sqrtf on every float of its domain.
* The kernel takes groups of eight rows untested where every lane is inside
  the image and tests and masks the others; sizes around its edges (one group,
  one wave of columns, a row remainder of every kind) and images that fill the
  whole square (non-zero border, no zero rows), are a single pixel, or hold
  negative, huge, infinite or NaN pixels must give the oracle's medians bit
  for bit, T0 bit for bit and T1..T5 within 1e-5 of FP64 where finite (the bar
  of the forward tests).
"""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import assert_same_indices, normwise_err
from tracetransform_amd import _lib, core

pytestmark = pytest.mark.gpu


def test_line_root_equals_sqrtf_on_its_domain(gpu):
    L = _lib.load()
    m, first = C.c_uint64(), C.c_uint32()
    for half in range(2):
        st = L.tt_testing_line_root(gpu.handle, half << 31, 1 << 31, C.byref(m),
                                    C.byref(first))
        assert st == _lib.TT_OK, L.tt_last_error()
        assert m.value == 0, hex(first.value)


def image(kind, n, rng):
    img = rng.random((n, n), dtype=np.float32)
    if kind == "full":        # non-zero up to the border
        return img + 0.25
    if kind == "inner":       # a zero border, as padding leaves it
        b = max(1, n // 6)
        out = np.zeros_like(img)
        out[b:-b, b:-b] = img[b:-b, b:-b]
        return out
    if kind == "pixel":
        out = np.zeros_like(img)
        out[n // 3, n // 2] = 0.5
        return out
    if kind == "signed":
        return img - 0.3
    out = np.zeros_like(img)
    b = max(1, n // 6)
    out[b:-b, b:-b] = img[b:-b, b:-b]
    out[n // 2, n // 2] = {"huge": 3e38, "inf": np.inf, "nan": np.nan}[kind]
    return out


@pytest.mark.parametrize("n", [3, 7, 8, 9, 12, 63, 64, 65, 70, 129, 200])
@pytest.mark.parametrize("kind", ["full", "inner", "pixel", "signed"])
def test_sizes_and_fills(oracle, gpu, n, kind):
    img = image(kind, n, np.random.default_rng(100 * n + len(kind)))
    A, step, codes = 24, 15.0, [0, 1, 2, 3, 4, 5]
    sino, aux = core.sinograms(torch.from_numpy(img).cuda(), A, step, codes, with_aux=True)
    g = sino.cpu().numpy()
    flat = np.ascontiguousarray(img).ravel()
    o, oaux = oracle.sinograms(flat, n, A, step, codes, nthreads=8)
    assert_same_indices("median_x", aux["median_x"].cpu(), oaux["med_x"])
    assert_same_indices("median_sqrt", aux["median_sqrt"].cpu(), oaux["med_s"])
    assert np.array_equal(g[0], o[0])
    d = oracle.sinograms_f64(flat, n, A, step, codes, oaux, nthreads=8, geometry=1)
    for t in range(1, 6):
        assert normwise_err(g[t], d[t]) <= 1e-5, t


@pytest.mark.parametrize("kind", ["huge", "inf", "nan"])
def test_extreme_pixels(oracle, gpu, kind):
    n, A, step = 75, 24, 15.0
    img = image(kind, n, np.random.default_rng(5))
    sino, aux = core.sinograms(torch.from_numpy(img).cuda(), A, step, [0, 1, 3], with_aux=True)
    o, oaux = oracle.sinograms(np.ascontiguousarray(img).ravel(), n, A, step, [0, 1, 3],
                               nthreads=8)
    assert_same_indices("median_x", aux["median_x"].cpu(), oaux["med_x"])
    assert_same_indices("median_sqrt", aux["median_sqrt"].cpu(), oaux["med_s"])
    assert np.array_equal(sino[0].cpu().numpy(), o[0], equal_nan=True)
    clean = np.isfinite(o[0]) & (np.abs(o[0]) < 1e30)  # lines without the pixel
    assert clean.sum() > 0.5 * clean.size
    for t in (1, 2):
        assert normwise_err(sino[t].cpu().numpy()[clean], o[t][clean]) <= 1e-4
