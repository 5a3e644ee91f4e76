"""The fit of a field under a mask against the FP64 oracle where its tiling
can go wrong: remainders of tiles and of eight-row loads, several chunks of
256 columns, more control points than one batch of rows holds, axes of one
voxel, runs of rows side by side in a workgroup.

Bound: numerator and denominator are FP32 sums of at most 64 rows, then of Z
columns, with factors rounded to FP32 (3 roundings a term), so each differs
from the exact sum by at most n 2^-24 times the sum of its terms' magnitudes,
n = 64 + Z + 3; the same fit of |field| gives that sum over the denominator."""
import numpy as np
import pytest

import oracle as O

CASES = [((3, 70, 44), (4, 7, 7)), ((2, 37, 257), (5, 6, 9)), ((2, 9, 600), (4, 4, 4)), ((40, 1, 1), (7, 4, 4)),
         ((1, 130, 3), (4, 60, 5)), ((5, 64, 16), (4, 67, 19)), ((9, 33, 31), (11, 11, 11)), ((2, 600, 2), (4, 5, 4)),
         ((1, 1, 513), (4, 4, 70))]


def _check(lib, dims, ncpt, fill):
    rng = np.random.default_rng(sum(dims))
    f = rng.standard_normal(dims).astype(np.float32)
    m = rng.random(dims) < fill
    f[~m] = np.nan  # not read into any sum
    lat = lib.fit_bspline3d(f, m, ncpt)
    g = np.where(m, f, 0).astype(np.float64)
    tol = (64 + dims[2] + 3) * 2.0**-24 * 2 * O.fit_bspline3d(np.abs(g), m, ncpt) + 1e-30
    assert np.all(np.abs(lat - O.fit_bspline3d(g, m, ncpt)) <= tol)


@pytest.mark.parametrize("fill", [0.0, 0.7])
@pytest.mark.parametrize("dims,ncpt", CASES)
def test_emulated(emu, dims, ncpt, fill):
    _check(emu, dims, ncpt, fill)


@pytest.mark.gpu
@pytest.mark.parametrize("fill", [0.0, 0.7])
@pytest.mark.parametrize("dims,ncpt", CASES)
def test_gpu(gpu, dims, ncpt, fill):
    _check(gpu, dims, ncpt, fill)


# More control points between a chunk's first and last column than it has
# columns.
MANY = [((2, 3, 100), (4, 4, 300)), ((2, 2, 256), (4, 4, 400)), ((3, 2, 300), (4, 4, 303)), ((2, 5, 259), (4, 6, 520)),
        ((2, 2, 513), (4, 4, 517)), ((2, 7, 300), (4, 5, 310))]


@pytest.mark.parametrize("dims,ncpt", MANY)
def test_many_control_points_emulated(emu, dims, ncpt):
    _check(emu, dims, ncpt, 0.7)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,ncpt", MANY)
def test_many_control_points_gpu(gpu, dims, ncpt):
    _check(gpu, dims, ncpt, 0.7)


# Spans of a quarter voxel and less: four spans in a row without a voxel leave
# a control point without support.
EMPTY = [((8, 8, 3), (11, 11, 19)), ((32, 32, 5), (11, 11, 35)), ((64, 64, 12), (67, 67, 67)), ((4, 4, 2), (4, 4, 15)),
         ((4, 4, 4), (4, 4, 35)), ((3, 4, 1), (4, 5, 300)), ((2, 5, 59), (4, 9, 300)), ((4, 3, 5), (4, 40, 5))]


@pytest.mark.parametrize("dims,ncpt", EMPTY)
def test_empty_spans_emulated(emu, dims, ncpt):
    _check(emu, dims, ncpt, 0.7)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,ncpt", EMPTY)
def test_empty_spans_gpu(gpu, dims, ncpt):
    _check(gpu, dims, ncpt, 0.7)
