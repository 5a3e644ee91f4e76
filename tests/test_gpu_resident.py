"""The resident kernel (one launch runs every volume's level/iteration loop,
a team of workgroups per volume) against the step path on the same inputs.

Both form the fit's and the field's sums in the same order with the same
roundings, so fields, lattices and normalised images are equal bit for bit;
only the FP64 convergence sums have another order (compared to 1e-9), which
moves no stop decision here."""
import numpy as np
import pytest

import parity_cases as PC

pytestmark = pytest.mark.gpu


def _both(gpu, vols, tile=0, **kw):
    try:
        gpu.set_tuning(path="steps", step_tile_voxels=tile, groups=1)
        ref = gpu.correct_batch(vols, **kw)
        # a workgroup count asks for the persistent kernel whatever the tile
        gpu.set_tuning(step_tile_voxels=tile, team_wgs_per_cu=1)
        out = gpu.correct_batch(vols, **kw)
        again = gpu.correct_batch(vols, **kw)
    finally:
        gpu.set_tuning(reset=True)
    for a, b, c in zip(ref, out, again):
        assert a["iterations"] == b["iterations"]
        assert (a["n_mask_full"], a["n_mask_work"]) == (b["n_mask_full"], b["n_mask_work"])
        assert np.allclose(a["last_cv"], b["last_cv"], rtol=1e-9, atol=1e-12)
        for k in ("log_bias", "normalized", "lattice"):
            assert np.array_equal(a[k], b[k]), k
            assert np.array_equal(b[k], c[k]), k  # reproducible
    return ref, out


def _vol(dims, seed, mask="f32"):
    im, m, _ = PC.small_phantom(dims, seed=seed)
    if mask == "none":
        return im, None
    return im, m.astype(np.uint8) if mask == "u8" else m


@pytest.mark.parametrize("precision", ["fp32", "bf16", "split_bf16"])
@pytest.mark.parametrize("dims,tile", [((17, 16, 16), 0), ((9, 33, 31), 0), ((20, 70, 45), 512), ((12, 130, 67), 1024),
                                       ((64, 15, 129), 0), ((3, 5, 200), 0), ((40, 48, 96), 2048)])
def test_shapes(gpu, precision, dims, tile):
    _both(gpu, [_vol(dims, 5)], tile, levels=3, max_iter=[5, 4, 3], fixed_iterations=True, precision=precision)


@pytest.mark.parametrize("mask", ["f32", "u8", "none"])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_uneven_batch_masks_and_shrinks(gpu, precision, mask):
    vols = [_vol(d, 30 + k, mask) for k, d in enumerate([(60, 52, 44), (34, 66, 50), (82, 38, 56), (97, 101, 89)])]
    _both(gpu, vols, levels=4, max_iter=[8, 6, 4, 2], threshold=0.001, precision=precision, shrink=[1, 1, 2, 3])


@pytest.mark.parametrize("kw", [dict(nbins=500), dict(nbins=16), dict(ncpt=(4, 5, 6), levels=2), dict(ncpt=(9, 16, 16), levels=1),
                                dict(max_iter=[3, 0, 2]), dict(fwhm=0.4, noise=0.1)])
def test_parameters(gpu, kw):
    p = dict(dict(levels=3, max_iter=[4, 3, 2], threshold=0.0005), **kw)
    _both(gpu, [_vol((44, 40, 36), 8)], **p)


def test_weighted_mask(gpu):
    im, m, _ = PC.small_phantom((48, 44, 40), seed=9)
    w = (m * np.linspace(0.2, 1.0, 40, dtype=np.float32)).astype(np.float32)
    _both(gpu, [(im, w)], levels=3, max_iter=[6, 5, 4], threshold=0.001, weighted_mask=True)


def test_degenerate_masks(gpu):
    im, m, _ = PC.small_phantom((30, 28, 26), seed=6)
    one = np.zeros_like(m)
    one[11, 13, 17] = 1
    split = m.copy()
    split[8:20] = 0  # slabs without foreground between two with
    ref, out = _both(gpu, [(im, np.zeros_like(m)), (np.full(im.shape, 100.0, np.float32), m), (im, one), (im, split)],
                     levels=2, max_iter=[4, 4], threshold=0.001)
    assert out[0]["n_mask_work"] == 0 and np.all(out[0]["log_bias"] == 0)


def test_more_volumes_than_compute_units(gpu):
    vols = [_vol((12 + k % 7, 14, 13), 100 + k) for k in range(40)] * 8
    _both(gpu, vols, levels=2, max_iter=[3, 3], threshold=0.001)


def test_large_single_volume_of_many_batches(gpu):
    """One workgroup holds more units than one LDS batch: few chunks, many
    slabs (a long x axis with small slabs in a batch of larger volumes)."""
    vols = [_vol((700, 16, 16), 3)] + [_vol((60, 70, 64), 40 + k) for k in range(24)]
    _both(gpu, vols, levels=2, max_iter=[3, 2], fixed_iterations=True, precision="bf16")
    _both(gpu, vols, levels=2, max_iter=[3, 2], fixed_iterations=True)


def test_covered_up_to_16_control_points_then_steps(gpu):
    """19 control points along y and z run on the step kernels: the default
    call equals them bit for bit."""
    v = [_vol((40, 36, 32), 4)]
    kw = dict(levels=4, max_iter=[2] * 4, ncpt=(5, 5, 5), fixed_iterations=True)
    a = gpu.correct_batch(v, **kw)
    try:
        gpu.set_tuning(path="steps")
        b = gpu.correct_batch(v, **kw)
    finally:
        gpu.set_tuning(reset=True)
    assert np.array_equal(a[0]["log_bias"], b[0]["log_bias"])


def _box(dims, z0, seed):
    """Tissue that the end of the field of view cuts off: foreground from z0
    to the last z, rows of several lengths."""
    rng = np.random.default_rng(seed)
    x, y, z = np.meshgrid(*(np.linspace(-1, 1, n) for n in dims), indexing="ij")
    im = np.where(x * x + y * y < 0.5, 200.0, 100.0) * np.exp(0.2 * (z + x * y)) + rng.normal(0, 4, dims)
    m = np.zeros(dims, np.uint8)
    m[1:-1, :, z0:] = 1
    m[:, dims[1] // 2:, :z0 + 4] = 0
    return im.astype(np.float32), m


@pytest.mark.parametrize("precision", ["fp32", "bf16", "split_bf16"])
@pytest.mark.parametrize("nz,z0", [(29, 12), (31, 12), (32, 12), (32, 28), (64, 12), (64, 28), (61, 44), (96, 76)])
def test_foreground_to_the_last_z(gpu, precision, nz, z0):
    _both(gpu, [_box((9, 37, nz), z0, nz)], levels=3, max_iter=[3, 3, 2], fixed_iterations=True, precision=precision)


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_no_fit_epsilon(gpu, precision):
    """With no term in the fit's denominator, control points without foreground
    have no value (0 / 0); the voxels that they do not touch keep theirs."""
    im, m = _box((40, 44, 48), 4, 2)
    m[:] = 0
    m[5:15, 11:22, 6:18] = 1  # whole spans of 5, 5.5 and 6 voxels
    kw = dict(levels=1, max_iter=[4], ncpt=(11, 11, 11), fixed_iterations=True, eps=0.0, precision=precision)
    try:
        gpu.set_tuning(path="steps")
        ref = gpu.correct_batch([(im, m)], **kw)[0]
    finally:
        gpu.set_tuning(reset=True)
    out = gpu.correct_batch([(im, m)], **kw)[0]
    assert np.isfinite(ref["log_bias"][m != 0]).all() and np.isnan(ref["lattice"]).any()
    for k in ("log_bias", "normalized", "lattice"):
        assert np.array_equal(out[k], ref[k], equal_nan=True), k


@pytest.mark.parametrize("precision", ["fp32", "bf16", "split_bf16"])
def test_any_number_of_workgroups(gpu, precision, monkeypatch):
    """The results do not depend on how many workgroups a call gets: teams of
    one workgroup a chunk, teams whose members have several, fewer workgroups
    than volumes; the same plan is used again with other teams."""
    vols = [_vol(d, 60 + k) for k, d in enumerate([(64, 60, 52), (18, 90, 47), (33, 20, 70), (5, 7, 9)])]
    kw = dict(levels=3, max_iter=[4, 3, 3], threshold=0.0005, precision=precision)
    ref = gpu.correct_batch(vols, **kw)
    for wgs in (1, 2, 3, 5, 8, 13, 30, 61, 256):
        monkeypatch.setenv("N4_RESIDENT_WGS", str(wgs))
        for a, b in zip(ref, gpu.correct_batch(vols, **kw)):
            assert a["iterations"] == b["iterations"] and a["last_cv"] == b["last_cv"], wgs
            assert (a["n_mask_full"], a["n_mask_work"]) == (b["n_mask_full"], b["n_mask_work"])
            for k in ("log_bias", "normalized", "lattice"):
                assert np.array_equal(a[k], b[k]), (wgs, k)


def test_handles_side_by_side(gpu):
    """Four threads with a handle and a stream each, large and small volumes
    and a batch: everyone gets the bits that it gets alone."""
    import ctypes as C
    import threading

    import n4amd

    jobs = [([_vol((150, 140, 130), 1)], "bf16"), ([_vol((120, 130, 140), 2)], "bf16"), ([_vol((40, 36, 33), 3)], "fp32"),
            ([_vol((60 + 9 * k, 50, 70 - 7 * k), 10 + k) for k in range(6)], "split_bf16")]
    state = []
    for vols, precision in jobs:
        lib = n4amd.Library(gpu.L, False)
        p = n4amd.default_params(levels=2, max_iter=[6, 5], threshold=0.0005, precision=precision)
        keep, arr = lib._batch_arrays(vols, p, True, None)
        stream = C.c_void_p()
        assert gpu.L.hipStreamCreateWithFlags(C.byref(stream), 1) == 0  # hipStreamNonBlocking
        state.append((lib, p, keep, arr, (n4amd.Report * len(vols))(), stream))

    def call(s):
        lib, p, _, arr, reports, stream = s
        return lib.L.n4_correct_batch(lib.h, arr, len(arr), C.byref(p), reports, stream)

    def results(s):
        return [k[i].download(np.float32, k[0]) for k in s[2] for i in (3, 5)]

    for s in state:
        assert call(s) == 0
    alone = [results(s) for s in state]
    status = [[] for _ in state]
    threads = [threading.Thread(target=lambda s=s, r=r: r.extend(call(s) for _ in range(12)))
               for s, r in zip(state, status)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s, ref, st in zip(state, alone, status):
        assert st == [0] * 12
        assert all(np.array_equal(a, b) for a, b in zip(ref, results(s)))
    for lib, _, keep, _, _, stream in state:
        for k in keep:
            for a in k[1:]:
                if a is not None:
                    a.free()
        assert gpu.L.hipStreamDestroy(stream) == 0 and lib.L.n4_destroy(lib.h) == 0


@pytest.mark.parametrize("dims,nvol,precision", [((128, 112, 16), 1, "bf16"), ((128, 112, 17), 1, "split_bf16"), ((200, 176, 5), 2, "fp32"),
                                                 ((200, 176, 6), 2, "fp32"), ((600, 240, 3), 3, "bf16"), ((600, 240, 4), 3, "fp32")])
def test_thin_grids_either_side_of_the_step_kernels(gpu, dims, nvol, precision):
    _both(gpu, [_vol(dims, 70 + k) for k in range(nvol)], levels=2, max_iter=[3, 2], fixed_iterations=True, precision=precision)


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_large_among_many_small(gpu, precision, monkeypatch):
    """As many volumes as compute units, a few of them large: teams for the
    large ones, the small ones in turn; with fewer workgroups as well."""
    small = [_vol((12 + k, 14, 13 + k), 200 + k) for k in range(5)]
    vols = (small * 50)[:250] + [_vol((90 - 4 * k, 88, 85), 210 + k) for k in range(6)]
    kw = dict(levels=2, max_iter=[3, 2], threshold=0.001, precision=precision)
    ref, out = _both(gpu, vols, **kw)
    monkeypatch.setenv("N4_RESIDENT_WGS", "40")
    for a, b in zip(out, gpu.correct_batch(vols, **kw)):
        assert a["iterations"] == b["iterations"]
        assert np.array_equal(a["log_bias"], b["log_bias"]) and np.array_equal(a["lattice"], b["lattice"])
