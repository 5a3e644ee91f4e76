"""Reconstruction tiles follow the size of the whole call, the limit of a
workgroup's LDS does not: long rows of few voxels are accepted at any size of
the volume and beside any neighbours (CPU build)."""
import numpy as np
import pytest

import n4amd
import oracle as O


@pytest.mark.parametrize("dims,ncpt", [((1100, 2000, 8), (4, 7, 4)), ((1000, 1100, 16), (4, 4, 9)), ((600, 3000, 12), (5, 4, 4)),
                                       ((560, 2100, 20), (4, 4, 19))])
def test_long_tiles_of_a_large_volume(emu, dims, ncpt):
    lat = np.random.default_rng(7).standard_normal(ncpt).astype(np.float32)
    out = emu.evaluate_bspline3d(lat, dims)
    wx, wy, wz = (_weights(n, c) for n, c in zip(dims, ncpt))
    xs = [0, dims[0] // 3, dims[0] - 1]
    want = np.einsum("xi,ijk,yj,zk->xyz", wx[xs], lat.astype(np.float64), wy, wz, optimize=True)
    # three FP32 contractions of four products each, weights rounded to FP32
    assert np.abs(out[xs] - want).max() <= 16 * 2.0**-24 * np.abs(lat).max() * 2


def _weights(n, c):
    w = np.zeros((n, c))
    pos = (np.arange(n) + 0.5) / (n / (c - 3))
    b = np.clip(np.floor(pos).astype(int), 0, c - 4)
    for a in range(n):
        w[a, b[a]:b[a] + 4] = O.cubic_bspline(pos[a] - b[a])
    return w


def test_refused_as_before(emu):
    """Rows too long for a workgroup at the smallest tile are refused at any
    size."""
    lat = np.zeros((4, 4, 4), np.float32)
    for dims in [(2, 4, 3300), (600, 7, 4200)]:
        with pytest.raises(n4amd.N4Error, match="LDS"):
            emu.evaluate_bspline3d(lat, dims)


def test_accepted_beside_a_large_neighbour(emu):
    """A volume of 8-voxel rows is corrected beside one that makes the tiles of
    the call larger, with the bits that it has alone."""
    rng = np.random.default_rng(3)
    vols = []
    for dims in [(32, 2040, 8), (260, 260, 260)]:
        im = (200 + 20 * rng.random(dims)).astype(np.float32)
        im[:, :, :1] = 0
        vols.append((im, None))
    kw = dict(levels=1, max_iter=[1], fixed_iterations=True, shrink=[8, 8])
    both = emu.correct_batch(vols, **kw)
    alone = emu.correct_batch(vols[:1], **dict(kw, shrink=[8]))
    assert np.array_equal(both[0]["log_bias"], alone[0]["log_bias"])
    assert np.array_equal(both[0]["normalized"], alone[0]["normalized"])


def _check_nonfinite(lib, dims, ncpt, bad, value):
    """Only the voxels whose span holds a non-finite control point are
    non-finite (at the very start of a span too, where its last factor is
    zero).  The others may be summed in another form: two sums of at most five
    products, each rounding within 2^-24 of the largest control point."""
    lat = np.random.default_rng(11).standard_normal(ncpt).astype(np.float32)
    clean = lib.evaluate_bspline3d(lat, dims)
    lat[bad] = value
    out = lib.evaluate_bspline3d(lat, dims)
    hit = np.ones(dims, bool)
    for d in range(3):
        n, c = dims[d], ncpt[d]
        b = np.clip(np.floor((np.arange(n) + 0.5) / (n / (c - 3))).astype(int), 0, c - 4)
        hit &= ((b <= bad[d]) & (bad[d] <= b + 3)).reshape([-1 if k == d else 1 for k in range(3)])
    assert not np.isfinite(out[hit]).any()
    assert np.abs(out[~hit] - clean[~hit]).max(initial=0) <= 10 * 2.0**-24 * np.abs(lat[np.isfinite(lat)]).max()


NONFINITE = [((5, 6, 30), (4, 4, 11), (2, 1, 9)), ((6, 5, 31), (4, 5, 11), (0, 4, 3)), ((4, 4, 64), (4, 4, 7), (1, 2, 0)),
             ((4, 9, 9), (4, 4, 11), (3, 3, 10)), ((3, 4, 45), (4, 4, 11), (1, 1, 5))]


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("dims,ncpt,bad", NONFINITE)
def test_nonfinite_control_point(emu, dims, ncpt, bad, value):
    _check_nonfinite(emu, dims, ncpt, bad, value)


@pytest.mark.gpu
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("dims,ncpt,bad", NONFINITE)
def test_nonfinite_control_point_gpu(gpu, dims, ncpt, bad, value):
    _check_nonfinite(gpu, dims, ncpt, bad, value)
