"""Rounding error of the 3 * 2^k lines along each axis, forward and inverse,
against transforms in extended precision.  Radix-3 and radix-2 stages with
every twiddle read from the table leave an RMS relative error of 0.34 eps
sqrt(log2 n) on random lines (1.5e-16 at 24 points, 2.1e-16 at 384); the bound
is 0.4 eps sqrt(log2 n), which twiddles formed as powers of one rounded root
(2.3e-16 and 3.1e-16 forward) do not meet."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rms(got, want):
    d = got.astype(np.clongdouble) - want
    return float(np.sqrt((np.abs(d) ** 2).sum() / (np.abs(want) ** 2).sum()))


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", [24, 48, 96, 192, 384])
def test_line(gpu, n, axis):
    import torch
    from ghost_amd import fftp
    shape = [4, 2, 2]  # the shortest rows a plan takes
    shape[axis] = n
    fwd = fftp.fftp3d_create_plan(shape, fftp.FFTW_REAL_TO_COMPLEX)
    inv = fftp.fftp3d_create_plan(shape, fftp.FFTW_COMPLEX_TO_REAL)
    rng = np.random.default_rng(401)
    err = np.zeros(2)
    reps = 40
    for _ in range(reps):
        r = rng.standard_normal(fwd.rshape)
        exact = np.fft.rfftn(r.astype(np.longdouble)).transpose(2, 1, 0)
        spec = np.ascontiguousarray(exact.astype(np.complex128))
        back = np.fft.irfftn(spec.astype(np.clongdouble).transpose(2, 1, 0), s=fwd.rshape, axes=(0, 1, 2)) * r.size
        c = torch.empty(fwd.cshape, dtype=torch.complex128, device="cuda")
        x = torch.empty(fwd.rshape, dtype=torch.float64, device="cuda")
        fftp.fftp3d_real_to_complex(fwd, torch.from_numpy(r).cuda(), c)
        fftp.fftp3d_complex_to_real(inv, torch.from_numpy(spec).cuda(), x)
        err += [rms(c.cpu().numpy(), exact) ** 2, rms(x.cpu().numpy(), back) ** 2]
    err = np.sqrt(err / reps)
    assert np.all(err < 0.4 * np.finfo(float).eps * np.sqrt(np.log2(n))), (n, axis, err)
