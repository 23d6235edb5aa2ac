"""Rows of one field whose x inverse shares a transform with a neighbouring
row: each keeps the accuracy it has alone.  A zero row beside a large one stays
exactly zero, a row 2^30 times smaller has an error relative to itself (0.4 eps
sqrt(log2 nx), the level of one line in test_gpu_line_rounding), a row that
overflows leaves its neighbour alone.  And whole transforms of random fields:
with rows transformed alone (their imaginary half of the rounding error
dropped) and one table root per radix-8 stage, c2r and r2c had the RMS errors
below, in units of 1e-16."""
import numpy as np
import pytest

from test_gpu_line_rounding import rms

pytestmark = pytest.mark.gpu

NX = [24, 32, 48, 64, 96, 128, 192, 256, 384, 512]


def c2r(spec, shape):
    import torch
    from ghost_amd import fftp
    p = fftp.fftp3d_create_plan(shape, fftp.FFTW_COMPLEX_TO_REAL)
    out = torch.full(p.rshape, 7.0, dtype=torch.float64, device="cuda")
    fftp.fftp3d_complex_to_real(p, torch.from_numpy(np.ascontiguousarray(spec)).cuda(), out)
    return out.cpu().numpy()


def row(a, nx):
    """The exact unnormalised inverse of a half row."""
    return np.fft.irfft(a.astype(np.clongdouble), n=nx) * nx


def half(nx, seed):
    """A half row of small whole numbers, its kx = 0 and nx/2 entries real."""
    rng = np.random.default_rng(seed)
    a = rng.integers(-500, 501, (nx // 2 + 1, 2)) @ np.array([1.0, 1.0j])
    a[0], a[-1] = a[0].real, a[-1].real
    return a


# x and y passes apart; both in one launch
@pytest.mark.parametrize("shape", [(n, 2, 3) for n in NX] + [(24, 64, 2), (64, 24, 3), (32, 48, 2), (48, 32, 2)])
def test_zero_rows(gpu, shape):
    nx, ny, nz = shape
    a = 1e6 * half(nx, 411)
    spec = np.broadcast_to(a[:, None, None], (nx // 2 + 1, ny, nz))  # only the row y = z = 0
    got = c2r(spec, shape)
    assert rms(got[0, 0], ny * nz * row(a, nx)) < 0.4 * np.finfo(float).eps * np.sqrt(np.log2(nx * ny * nz))
    got[0, 0] = 0.0
    assert np.all(got == 0.0)


@pytest.mark.parametrize("small", [0, 1])
@pytest.mark.parametrize("nx", NX)
def test_rows_of_very_different_size(gpu, nx, small):
    a, b = half(nx, 421), 2.0 ** -30 * half(nx, 422)
    if small == 0:
        a, b = b, a
    spec = np.zeros((nx // 2 + 1, 2, 2), dtype=complex)
    spec[:, 0, 0], spec[:, 1, 0] = a + b, a - b  # rows 2 a and 2 b, exact sums
    got = c2r(spec, (nx, 2, 2))
    for z in range(2):
        for y, want in enumerate((2 * row(a, nx), 2 * row(b, nx))):
            assert rms(got[z, y], want) < 0.4 * np.finfo(float).eps * np.sqrt(np.log2(nx)), (z, y)


@pytest.mark.parametrize("nx", NX)
def test_a_row_that_overflows(gpu, nx):
    spec = np.zeros((nx // 2 + 1, 2, 2), dtype=complex)
    spec[:, :, 0] = 1.2e308 * (half(nx, 431) / 1000.0).real[:, None] + 1.2e308  # y = 0 overflows, y = 1 cancels
    got = c2r(spec, (nx, 2, 2))
    assert not np.any(np.isfinite(got[:, 0])) and np.all(got[:, 1] == 0.0)


BEFORE = {(32, 32, 32): (3.64, 3.42), (64, 64, 64): (4.32, 4.00), (128, 128, 128): (5.13, 4.63),
          (512, 64, 32): (4.59, 4.14), (256, 128, 16): (4.42, 4.07), (24, 24, 24): (2.79, 2.74),
          (48, 48, 48): (3.10, 3.02), (96, 96, 96): (3.40, 3.30), (192, 192, 48): (3.48, 3.36),
          (384, 96, 48): (3.48, 3.32)}


@pytest.mark.parametrize("shape", BEFORE)
def test_whole_transforms(gpu, shape):
    import torch
    from ghost_amd import fftp
    f = fftp.fftp3d_create_plan(shape, fftp.FFTW_REAL_TO_COMPLEX)
    r = np.random.default_rng(0).standard_normal(f.rshape)
    exact = np.fft.rfftn(r.astype(np.longdouble)).transpose(2, 1, 0)
    spec = exact.astype(np.complex128)
    back = np.fft.irfftn(spec.astype(np.clongdouble).transpose(2, 1, 0), s=f.rshape, axes=(0, 1, 2)) * r.size
    c = torch.empty(f.cshape, dtype=torch.complex128, device="cuda")
    fftp.fftp3d_real_to_complex(f, torch.from_numpy(r).cuda(), c)
    got = rms(c.cpu().numpy(), exact), rms(c2r(spec, shape), back)
    for g, before in zip(got, BEFORE[shape]):
        assert g < 1.01e-16 * before, got
