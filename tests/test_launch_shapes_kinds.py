"""Launch shapes of the grouped updates, the small planes, the x passes by row
count and the y and z passes on schedules of their own, as in
test_launch_shapes: computed on the host by the functions the launchers call,
for every line length, tile request and both LDS limits.  The grouped updates
and the small planes are only taken where a device has their LDS (-3: the
launcher takes the other kernels)."""
import pytest

from test_launch_shapes import LIMITS, ROW_BOUND, SIZES, TILE_BOUND, WANTS, X2, shape

ROWS = [1, 2, 63, 64, 65, 2303, 2304, 2305, 4607, 4608, 4609, 9215, 9216, 9217, 18432, 18433, 147456, 147457, 1 << 20]


@pytest.mark.parametrize("kind,groups,bound", [(5, 3, 768), (6, 3, 768), (7, 4, 512)])
def test_grouped_updates(kind, groups, bound):
    for n in SIZES:
        for nlines in (1, 2, 3, 5, 8, 17, 33, 1024):
            for want in WANTS:
                for limit in LIMITS:
                    rc, L, block, lds, T = shape(kind, n, nlines, want, limit)
                    one = groups * (n + n // 8 + 1) * 16  # one line of every component
                    assert rc == (0 if one <= limit else -3), (kind, n, nlines, want, limit)
                    if rc:
                        continue
                    assert L >= 1 and L & (L - 1) == 0 and L <= 32
                    assert L <= max(1, nlines) and (want < 2 or L <= want)
                    assert block == groups * L * T <= bound and lds == L * one


def test_small_planes():
    for nx in SIZES:
        for ny in SIZES:
            rc, rows, block, lds, T = shape(8, nx, ny, 0, 163840)
            if nx not in (24, 32, 48, 64) or ny not in (24, 32, 48, 64):
                assert rc == -1
                continue
            assert rc == 0 and block == ROW_BOUND == rows * T
            assert lds == (rows * (nx + nx // 8 + 1) + (nx // 2 + 1) * (ny + ny // 8 + 1)) * 16 <= 163840
            assert shape(8, nx, ny, 0, 65536)[0] == (0 if lds <= 65536 else -3)
    assert shape(8, 64, 64, 0, 65536)[0] == -3  # 76 KB


@pytest.mark.parametrize("kind", [10, 11])
def test_row_passes_by_row_count(kind):
    for n in SIZES:
        for rows in ROWS:
            for limit in LIMITS:
                rc, R, block, lds, T = shape(kind, n, rows, 0, limit)
                if kind == 10 and n not in X2:
                    assert rc == -1
                    continue
                assert rc == 0 and R >= 1 and block == R * T <= ROW_BOUND
                assert lds == R * (n + n // 8 + 1) * 16 <= limit
                # up to 2304 wavefronts in blocks of one, then whole blocks
                assert block == max(T, 64 if rows * T <= 64 * 2304 else ROW_BOUND)


@pytest.mark.parametrize("kind,lanes", [(12, {96: 8, 192: 16, 384: 32}), (13, {192: 16, 384: 32}),
                                        (14, {192: 16, 384: 32})])
def test_passes_on_other_schedules(kind, lanes):
    for n in SIZES:
        for nlines in (1, 3, 8, 33, 1024):
            for want in WANTS:
                for limit in LIMITS:
                    rc, L, block, lds, T = shape(kind, n, nlines, want, limit)
                    assert rc == 0 and T == lanes.get(n, shape(0, n, nlines, want, limit)[4])
                    assert L >= 1 and L & (L - 1) == 0 and L <= min(32, max(1, nlines))
                    assert block == L * T <= TILE_BOUND and lds == L * (n + n // 8 + 1) * 16 <= limit


def test_updates_keep_the_large_launches_schedule():
    """Four points per lane for MHD on 32 to 512 points and HD on 512, as the
    updates that take one component after another; else the default schedule."""
    for n in SIZES:
        low = n in (32, 64, 128, 256, 512)
        default = shape(0, n, 8, 1, 163840)[4]
        assert shape(5, n, 8, 1, 163840)[4] == (128 if n == 512 else default)
        assert shape(6, n, 8, 1, 163840)[4] == (n // 4 if low else default)
        assert shape(7, n, 8, 1, 163840)[4] == default


def test_one_field_per_block_ends_earlier_on_long_lines():
    """Up to 192 points one limit, beyond a volume of lines (5 to 40% slower
    above it at 256 to 1024 points), never below a tile for most CUs."""
    for n in SIZES:
        z, y = shape(15, n, 1, 0, 163840), shape(16, n, 1, 0, 163840)
        assert z[0] == y[0] == 0
        assert z[1] == (3328 if n <= 192 else max(384, 1408 * 192 // n))
        assert y[1] == {384: 2112, 1024: 512}.get(n, 3328)


def test_long_y_inverses_split_where_it_gains():
    for n in SIZES:
        for nf in (1, 3, 6, 9):
            for lines in (3329, 9999, 10000, 11008, 16416, 19999, 20000, 22016, 49536):
                want = lines >= 10000 and (n <= 96 or n == 192 or
                                           (n in (256, 384) and nf >= 6 and lines >= 20000))
                assert shape(17, n, lines, nf, 163840)[:2] == (0, int(want))
                assert shape(18, n, lines, nf, 163840)[:2] == (0, int(lines >= 10000 and n != 512))
