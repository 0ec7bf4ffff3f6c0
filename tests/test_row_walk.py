"""Division of the 256 x 256 tiles of row groups among the workgroups of an XCD, as the kernels compute it (run on the host)."""
import ctypes

import pytest

from mslk_amd import _lib


def _entry(tiles, wgs, worker, pass_):
    piece, pieces = ctypes.c_int(), ctypes.c_int()
    entry = _lib.lib().mslk_amd_debug_row_walk(tiles, wgs, worker, pass_, ctypes.byref(piece), ctypes.byref(pieces))
    assert entry >= -1
    return entry, piece.value, pieces.value


def _walk(tiles, wgs, worker):
    """All entries of one workgroup, which come without a gap."""
    out = []
    for pass_ in range(tiles // wgs + 3):
        entry = _entry(tiles, wgs, worker, pass_)
        if entry[0] < 0:
            break
        out.append(entry)
    assert all(_entry(tiles, wgs, worker, p)[0] < 0 for p in range(len(out), tiles // wgs + 4))
    return out


@pytest.mark.parametrize("wgs", [1, 2, 3, 4, 5, 6, 8, 31, 32])
def test_every_tile_is_computed_once(wgs):
    for tiles in list(range(0, 3 * wgs + 2)) + [7 * wgs - 1, 7 * wgs, 9 * wgs + wgs // 4, 9 * wgs + wgs // 4 + 1]:
        seen = {}
        for worker in range(2 * wgs):
            for entry, piece, pieces in _walk(tiles, wgs, worker):
                assert (entry, piece) not in seen and piece < pieces
                seen[entry, piece] = pieces
        assert sorted({e for e, _ in seen}) == list(range(tiles))
        for (entry, _), pieces in seen.items():
            assert all((entry, p) in seen for p in range(pieces))


@pytest.mark.parametrize("rows", [2, 3, 4])
@pytest.mark.parametrize("wgs", [4, 8, 16, 30, 31, 32])
def test_ragged_tiles_of_panels_are_shared_out(rows, wgs):
    """Panels of `rows` row tiles whose last is ragged: over twelve passes every workgroup gets its even share of them, give or take
    two (where its entries go round the end of a pass the sequence breaks)."""
    passes = 12
    for worker in range(wgs):
        ragged = sum(entry % rows == rows - 1 for entry, _, _ in _walk(passes * wgs, wgs, worker))
        assert passes // rows - 2 <= ragged <= passes // rows + 2, (worker, ragged)
