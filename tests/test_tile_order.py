"""The order in which the blocks of a z or y pass take their tiles.  Blocks go to
the 8 XCDs by linear id mod 8: every tile is taken once, neighbouring tiles of a
pair share an XCD, and the tiles that a pruned pass keeps are spread evenly: the
outer thirds of ky in the z passes (rows of 16, 32 and 64 tiles among them), the
lower two thirds of kx in the y passes."""
import ctypes as C

import numpy as np
import pytest

import ghost_amd


def order(gx, rows, spread=1):
    t = (C.c_int * (gx * rows))()
    assert ghost_amd.load().ghx_tile_order(gx, rows, spread, t) == 0
    return np.array(t)


def xcds(gx, rows, spread=1):
    x = np.empty(gx * rows, int)
    x[order(gx, rows, spread)] = np.arange(gx * rows) % 8
    return x


@pytest.mark.parametrize("spread", [0, 1])
@pytest.mark.parametrize("rows", [1, 2, 7, 33, 129])
@pytest.mark.parametrize("gx", [1, 2, 3, 5, 8, 12, 15, 16, 17, 24, 32, 33, 48, 64, 128, 256])
def test_every_tile_once(gx, rows, spread):
    assert np.array_equal(np.sort(order(gx, rows, spread)), np.arange(gx * rows))


@pytest.mark.parametrize("spread", [0, 1])
@pytest.mark.parametrize("gx", [5, 16, 24, 48, 64])
def test_pairs_share_an_xcd(gx, spread):
    x = xcds(gx, 33, spread)
    full = len(x) & ~15
    assert np.array_equal(x[0:full:2], x[1:full:2])


def even(load):
    """Within an eighth of the mean beside a few tiles."""
    return load.max() <= 1.125 * load.mean() + 4


@pytest.mark.parametrize("nxh", [43, 65, 129, 257])
@pytest.mark.parametrize("ny,lines", [(64, 4), (128, 4), (128, 8), (192, 4), (256, 4), (256, 8), (384, 4), (384, 8),
                                      (512, 4), (512, 8), (1024, 4), (1024, 8)])
def test_kept_tiles_of_z_passes(nxh, ny, lines):
    nt = ny // lines
    assert nt % 16 == 0
    ky = np.minimum(np.arange(ny), ny - np.arange(ny))
    on = np.add.reduceat(ky <= ny / 3, np.arange(0, ny, lines)) > 0
    kept = xcds(nt, nxh).reshape(nxh, nt)[:nxh * 2 // 3, on]
    assert even(np.bincount(kept.ravel(), minlength=8))


@pytest.mark.parametrize("nx", [24, 32, 64, 96, 128, 192, 256, 384, 512])
@pytest.mark.parametrize("nz", [24, 32, 48, 64, 128, 192, 256, 512])
def test_kept_tiles_of_y_passes(nx, nz):
    nt = (nx // 2 + 1 + 7) // 8
    on = np.arange(nt) * 8 <= nx // 3
    kept = xcds(nt, nz, 0).reshape(nz, nt)[:, on]
    assert even(np.bincount(kept.ravel(), minlength=8))


def test_bad_arguments():
    lib = ghost_amd.load()
    t = (C.c_int * 4)()
    assert lib.ghx_tile_order(0, 1, 1, t) == lib.ghx_tile_order(1, 0, 1, t) == lib.ghx_tile_order(1, 1, 1, None) == -1
