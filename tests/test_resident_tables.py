"""The resident kernel's factor tables (res_tables of the host emulation
build, the code that the device runs) hold a value wherever its loops read
one.  The LDS starts out as NaN bytes, as it may on the device.

A unit of the foreground starts at a multiple of four (zlo) and is read in
tiles of 16 z up to the one that holds its last foreground voxel, so a tile
may start at any multiple of four below Z and reaches 15 past its start; rows
come in blocks of 16 from a multiple of 16."""
import ctypes as C

import numpy as np
import pytest

AXIS = np.dtype([("w", "<f4", 4), ("p", "<f4", 4), ("q", "<f4", 4), ("b", "<i4"), ("pad", "<i4", 3)])


def _axis(n, c):
    pos = (np.arange(n) + 0.5) / (n / (c - 3))
    b = np.clip(np.floor(pos).astype(int), 0, c - 4)
    t = pos - b
    w = np.stack([(1 - t) ** 3, 3 * t ** 3 - 6 * t ** 2 + 4, -3 * t ** 3 + 3 * t ** 2 + 3 * t + 1, t ** 3], 1) / 6
    a = np.zeros(n, AXIS)
    a["w"], a["q"], a["b"] = w, w ** 2, b
    a["p"] = w ** 3 / (w ** 2).sum(1, keepdims=True)
    return a


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("ncp", [4, 11, 16])
@pytest.mark.parametrize("Y,Z", [(1, 1), (16, 29), (15, 30), (33, 31), (40, 32), (48, 64), (17, 61), (96, 96), (70, 44),
                                 (31, 33), (64, 160), (130, 67)])
def test_every_entry_read_is_filled(emu, prec, ncp, Y, Z):
    axy, axz = _axis(Y, ncp), _axis(Z, ncp)
    lds = np.full(160 * 1024, 0xFF, np.uint8)
    off = np.zeros(9, np.uint32)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)
    fill = emu.L.n4emu_resident_tables
    fill.restype = C.c_int64
    for kf in (2, 1):  # the denominator's tables, then the iterations'
        n = fill(ptr(axy), Y, ptr(axz), Z, ncp, prec, kf, ptr(lds), C.c_int64(lds.size), ptr(off))
        assert 0 < n <= lds.size
    zw, zb, wy, pz, pzl, py, pyl, pzs, pys = (int(o) for o in off)

    def at(start, dtype, index):
        return lds[start:n - (n - start) % np.dtype(dtype).itemsize].view(dtype)[index]

    starts = np.arange(0, Z, 4)
    z = (starts[:, None] + np.arange(16)).reshape(-1)
    y = (np.arange(0, Y, 16)[:, None] + np.arange(16)).reshape(-1)
    # evaluation: the spans of a tile bound a loop; rows past the grid count nothing
    b = at(zb, np.int32, z)
    assert b.min() >= 0 and b.max() <= ncp - 4
    assert np.array_equal(b, axz["b"][np.minimum(z, Z - 1)])
    want = np.where((z < Z)[:, None], axz["w"][np.minimum(z, Z - 1)], 0).astype(np.float32)[:, [1, 0, 2, 3]]
    assert np.array_equal(at(zw, np.float32, 4 * z[:, None] + np.arange(4)), want)
    assert np.isfinite(at(wy, np.float32, 16 * y[:, None] + np.arange(16))).all()
    # fit: the control points' rows, including what a row's last reads take past it
    c = np.arange(16)[:, None]
    if prec == 0:
        for tab, st, pos in ((pz, pzs, z), (py, pys, y)):
            assert np.isfinite(at(tab, np.float32, (4 * c + pos % 4) * st + pos // 4)).all()
    else:
        blocks = np.arange(32 * ((z.max() + 32) // 32))  # blocks of 32 z from z = 0
        for tab, st, pos in ((pz, pzs, blocks), (pzl, pzs, blocks), (py, pys, y), (pyl, pys, y)):
            half = at(tab, np.uint16, c * st + pos).astype(np.uint32) << 16
            assert np.isfinite(half.view(np.float32)).all()
