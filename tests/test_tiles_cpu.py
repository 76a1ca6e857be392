"""Tile tables of the smaller tile shapes (host side of the sorted list)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import capi


def _lib():
    lib = capi.lib()
    lib.rumdx_tile_table_shaped.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
    lib.rumdx_tile_shape.argtypes = [C.c_void_p]
    return lib


@pytest.mark.parametrize("shape,edge", [(0, (4, 4, 4)), (1, (4, 4, 2)), (2, (4, 2, 2)), (3, (2, 2, 2))])
@pytest.mark.parametrize("nc_list", [[27, 27, 27], [6, 7, 5], [9, 12, 10]])
def test_smaller_tiles_are_contiguous_rank_ranges(nc_list, shape, edge):
    lib = _lib()
    nc = np.array(nc_list, dtype=np.int32)
    ncells = int(nc.prod())
    rank = np.zeros(ncells, dtype=np.uint32)
    assert lib.rumdx_cell_rank_table(nc, rank) == 0
    nt = lib.rumdx_tile_table_shaped(nc.ctypes.data, None, shape, None, None)
    assert nt == int(np.prod([-(-n // e) for n, e in zip(nc, edge)]))
    first = np.zeros(nt + 1, dtype=np.uint32)
    origin = np.zeros(nt, dtype=np.uint32)
    assert lib.rumdx_tile_table_shaped(nc.ctypes.data, rank.ctypes.data, shape, first.ctypes.data, origin.ctypes.data) == nt
    assert first[0] == 0 and first[-1] == ncells and np.all(origin >> 30 == shape)
    inv = np.argsort(rank)  # rank -> linear cell
    for t in range(nt):
        cells = inv[first[t]:first[t + 1]]
        at = np.stack([cells % nc[0], (cells // nc[0]) % nc[1], cells // (nc[0] * nc[1])])
        o = np.array([origin[t] & 1023, (origin[t] >> 10) & 1023, (origin[t] >> 20) & 1023])
        own = np.minimum(edge, nc - o)
        assert cells.size == own.prod()
        assert np.array_equal(at.min(axis=1), o) and np.array_equal(at.max(axis=1), o + own - 1)


def test_tile_shape_rule():
    """Small grids take small tiles, grids with 4^3 tiles enough keep them."""
    lib = _lib()
    grids = [np.array([n] * 3, np.int32) for n in (5, 13, 20, 21, 27, 36, 68)]
    got = [lib.rumdx_tile_shape(g.ctypes.data) for g in grids]
    assert got == sorted(got, reverse=True) and got[0] == 3 and got[-1] == 0
    assert lib.rumdx_tile_table_shaped(grids[0].ctypes.data, None, 4, None, None) == -1
