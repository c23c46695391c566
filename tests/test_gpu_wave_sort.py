"""GPU tests of the one-wave circus kernel and of the wave sort behind P2, T6
and T7 at its edges: every network
width (64 keys and powers of two up to 2048) from one row short to one row
over, signed values, ties, both zeros, infinities, and NaN columns.  Ranks
and values are the oracle's exactly; a column with a NaN has a NaN sum, which
no prefix reaches: the last position, its value the largest with a positive
NaN above everything.
"""
import numpy as np
import pytest
import torch

from helpers import assert_same_indices, normwise_err
from tracetransform_amd import core

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 63, 64, 65, 127, 128, 129, 255, 257, 511, 512, 513, 1023, 1025, 2047, 2048]


def p2(cols):
    circ, rank = core.circus(torch.from_numpy(cols[None]).cuda(), [(2,)], with_p2_rank=True)
    return circ[0, 0].cpu().numpy(), rank[0, 0].cpu().numpy()


@pytest.mark.parametrize("n", SIZES)
def test_p2_edges(oracle, gpu, n):
    rng = np.random.default_rng(n)
    cols = np.stack([
        rng.random(n),
        rng.random(n) - 0.5,
        np.round(rng.random(n) * 8) / 8,                     # ties
        np.where(rng.random(n) < 0.5, 0.0, -0.0) + np.round(rng.random(n)),
        -np.arange(n, dtype=np.float64),                     # descending
        np.where(np.arange(n) == n // 2, np.inf, rng.random(n)),
        np.full(n, 1e-42),                                   # denormal
        np.zeros(n),
    ]).astype(np.float32)
    got, rank = p2(cols)
    want, aux = oracle.circus(cols, n, len(cols), [(2,)])
    assert_same_indices("rank", rank, aux["p2_rank"][0])
    assert np.array_equal(got, want[0])


@pytest.mark.parametrize("n", [2, 3, 64, 512, 513, 1024, 1025, 2048, 2049, 2730])
def test_p1_p2_p3_key_widths(oracle, gpu, n):
    # the kernel's three key widths and the longer columns' own kernel, the
    # functionals in any order and repeated
    rng = np.random.default_rng(n)
    cols = (rng.random((5, n)) * 3).astype(np.float32)
    pf = [(3,), (1,), (2,), (1,), (3,)]
    got, rank = core.circus(torch.from_numpy(cols[None]).cuda(), pf, with_p2_rank=True)
    _, aux = oracle.circus(cols, n, 5, pf)
    want = oracle.circus_f64(cols, n, 5, pf, aux["p2_src"], geometry=1)
    got = got[0].cpu().numpy()
    assert_same_indices("rank", rank[0, 2].cpu(), aux["p2_rank"][2])
    for q in range(len(pf)):
        assert normwise_err(got[q], want[q]) <= 1e-5, pf[q]
    assert np.array_equal(got[0], got[4]) and np.array_equal(got[1], got[3])


@pytest.mark.parametrize("n", [5, 64, 300, 1500])
def test_p2_nan_columns(gpu, n):
    rng = np.random.default_rng(n)
    cols = rng.random((3, n)).astype(np.float32)
    cols[0, n // 3] = np.nan
    cols[1, n - 1] = np.nan
    cols[2, 0] = -np.float32(np.nan)
    assert np.signbit(cols[2, 0])
    got, rank = p2(cols)
    assert (rank == n - 1).all()
    assert np.isnan(got[0]) and np.isnan(got[1])
    assert got[2] == np.nanmax(cols[2])


@pytest.mark.parametrize("side", [60, 64, 90, 130, 182, 260, 364, 520])
def test_t6_t7_widths(oracle, gpu, side):
    # an image that fills its square: tails of every length up to the side
    n, A, step = side, 6, 60.0
    img = np.random.default_rng(side).random((n, n), dtype=np.float32)
    img[:, ::7] = 0.0
    sino, aux = core.sinograms(torch.from_numpy(img).cuda(), A, step, [6, 7], with_aux=True)
    o, oaux = oracle.sinograms(np.ascontiguousarray(img).ravel(), n, A, step, [6, 7],
                               nthreads=8)
    assert_same_indices("t6_rank", aux["t6_rank"].cpu(), oaux["t6_rank"])
    assert_same_indices("t6_src", aux["t6_src"].cpu(), oaux["t6_src"])
    assert_same_indices("t7_rank", aux["t7_rank"].cpu(), oaux["t7_rank"])
    assert_same_indices("t7_src", aux["t7_src"].cpu(), oaux["t7_src"])
    assert np.array_equal(sino.cpu().numpy(), o)


@pytest.mark.parametrize("n", [3, 64, 513, 2048, 2049])
@pytest.mark.parametrize("codes", [[1, 0], [0, 3], [0, 3, 1, 0], [2, 0, 1], [0, 2]])
def test_lists_with_hermite(oracle, gpu, n, codes):
    # Hermite entries with P1 and P3 in the workgroup kernel, and P1..P3 in the
    # wave kernel beside them where P2 is in the list
    rng = np.random.default_rng(10 * n + len(codes))
    cols = (rng.random((5, n)) * 3).astype(np.float32)
    pf = [(c,) if c else (0, 1 + q, n // 2) for q, c in enumerate(codes)]
    got, rank = core.circus(torch.from_numpy(cols[None]).cuda(), pf, with_p2_rank=True)
    _, aux = oracle.circus(cols, n, 5, pf)
    want = oracle.circus_f64(cols, n, 5, pf, aux["p2_src"], geometry=1)
    got = got[0].cpu().numpy()
    if 2 in codes:
        q = codes.index(2)
        assert_same_indices("rank", rank[0, q].cpu(), aux["p2_rank"][q])
    for q in range(len(pf)):
        assert normwise_err(got[q], want[q]) <= 1e-5, pf[q]


@pytest.mark.parametrize("n", [2, 3, 64, 65, 66, 449, 512, 513, 514, 577, 1025, 1026, 2047, 2048])
def test_p1_rows(gpu, n):
    # whole numbers: every sum is exact, a term left out or taken twice shows
    x = np.random.default_rng(n).integers(-40, 41, (3, n)).astype(np.float32)
    got = core.circus(torch.from_numpy(x[None]).cuda(), [(1,)])[0, 0].cpu().numpy()
    assert np.array_equal(got, np.abs(np.diff(x, axis=1)).sum(axis=1))


@pytest.mark.parametrize("n", [5, 67, 68, 69, 132, 133, 260, 261, 516, 517, 900, 1028, 1029, 1500,
                               2047, 2048])
def test_t6_t7_values_without_sources(oracle, gpu, n):
    # T6 and T7 as a caller without index outputs gets them (T7 sorted by its
    # values alone), together and each alone.  Two bright rows put the medians
    # at the lines' starts: tails of 64 keys and powers of two up to 2048, one
    # more and one less, distinct values in half of the columns and ties in the
    # others, trailing zeros and zeros in between.
    rng = np.random.default_rng(n)
    img = rng.random((n, n), dtype=np.float32)
    img[::2] = np.round(img[::2] * 64) / 64
    img[:, 5::11] = 0.0
    img[:, -2:] = 0.0
    img[:, :2] = np.float32(n) ** 2
    A, step = 3, 20.0
    t = torch.from_numpy(img).cuda()
    o, oaux = oracle.sinograms(img.ravel(), n, A, step, [6, 7], nthreads=8)
    if n > 60:
        assert (n - oaux["med_x"][0] >= n - 2).mean() > 0.9  # long tails at 0 degrees
    both = core.sinograms(t, A, step, [6, 7]).cpu().numpy()
    assert np.array_equal(both, o)
    assert np.array_equal(core.sinograms(t, A, step, [7]).cpu().numpy()[0], o[1])
    assert np.array_equal(core.sinograms(t, A, step, [6]).cpu().numpy()[0], o[0])
