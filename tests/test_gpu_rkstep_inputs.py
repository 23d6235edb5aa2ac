"""The substeps on caller fields, whose passes skip what lies outside the
dealias set when a kernel finds the input zero there: dealiased input, input
with one mode outside the set in the last field, and input with every mode
filled; dense forcing; output buffers that held something else.  One ord = 1
step against the oracle, relative L2 1e-12, exact zeros outside the set."""
import numpy as np
import pytest

from test_gpu_parity import grids, rand_spec, rel, to_gpu, to_np

pytestmark = pytest.mark.gpu

# cubic, uneven, a row length without the two-for-one x kernels, and the
# 512-point schedules of the y and z passes
SHAPES = [((32, 32, 32), False, (1, 1, 1)), ((24, 16, 48), True, (1.0, 1.0, 0.5)), ((20, 24, 6), False, (1, 1, 1)),
          ((16, 512, 8), False, (1, 1, 1)), ((16, 8, 512), False, (1, 1, 1))]


def kept(shape, arb):
    nx, ny, nz = shape
    i, j, k = np.arange(nx // 2 + 1), np.fft.fftfreq(ny, 1.0 / ny), np.fft.fftfreq(nz, 1.0 / nz)
    i = np.where(i < nx // 2, i, i - nx)
    anis = arb or nx != ny or ny != nz
    s = (1.0 / nx ** 2, 1.0 / ny ** 2, 1.0 / nz ** 2) if anis else (1.0, 1.0, 1.0)
    kn2 = s[0] * (i ** 2)[:, None, None] + s[1] * (j ** 2)[None, :, None] + s[2] * (k ** 2)[None, None, :]
    lim = 1.0 / 9.0 if anis else nx * nx / 9.0
    return (kn2 <= lim) & (kn2 > 0)


def fields(og, mask, n, seed, how):
    out = [rand_spec(og, seed + q) for q in range(n)]
    if how != "full":
        out = [np.where(mask, x, 0.0) for x in out]
    if how == "one":
        at = tuple(np.argwhere(~mask)[-1])
        out[-1][at] = 0.25 - 0.5j
    return out


def check(got, want, mask):
    for k, (a, b) in enumerate(zip(got, want)):
        a = to_np(a)
        assert rel(a, b) < 1e-12, k
        assert not np.any(a[~mask][np.asarray(b)[~mask] == 0.0]), k


@pytest.mark.parametrize("how", ["clean", "one", "full"])
@pytest.mark.parametrize("shape,arb,L", SHAPES)
def test_hd(gpu, shape, arb, L, how):
    import torch
    g, og = grids(shape, arb, L)
    m = kept(shape, arb)
    v, f = fields(og, m, 3, 101, how), fields(og, m, 3, 111, "full")
    V, F = [to_gpu(x) for x in v], [to_gpu(x) for x in f]
    for force in (None, f):
        out = [torch.full_like(x, 7.0) for x in V]
        g.hd_rkstep2(1, 1e-3, 4e-3, V, V, None if force is None else F, out)
        want = [x.copy() for x in v]
        og.hd_step(want, 1e-3, 4e-3, f=force, ord=1)
        check(out, want, m)


@pytest.mark.parametrize("how", ["clean", "one", "full"])
@pytest.mark.parametrize("shape,arb,L", SHAPES)
def test_mhd(gpu, shape, arb, L, how):
    import torch
    g, og = grids(shape, arb, L)
    m = kept(shape, arb)
    s, f = fields(og, m, 6, 121, how), fields(og, m, 6, 131, "full")
    S, F = [to_gpu(x) for x in s], [to_gpu(x) for x in f]
    out = [torch.full_like(x, 7.0) for x in S]
    g.mhd_rkstep2(1, 1e-3, 4e-3, 5e-3, S, S, F[:3], F[3:], out)
    v, a = [x.copy() for x in s[:3]], [x.copy() for x in s[3:]]
    og.mhd_step(v, a, 1e-3, 4e-3, 5e-3, f=f[:3], m=f[3:], ord=1)
    check(out, v + a, m)


@pytest.mark.parametrize("how", ["clean", "one", "full"])
@pytest.mark.parametrize("shape,arb,L", SHAPES)
def test_bouss(gpu, shape, arb, L, how):
    """The temperature's mean is carried, so it may be non-zero in clean input."""
    import torch
    g, og = grids(shape, arb, L)
    m = kept(shape, arb)
    s, f = fields(og, m, 4, 141, how), fields(og, m, 4, 151, "full")
    s[3][0, 0, 0] = 3.0
    S, F = [to_gpu(x) for x in s], [to_gpu(x) for x in f]
    out = [torch.full_like(x, 7.0) for x in S]
    g.bouss_rkstep2(1, 1e-3, 4e-3, 5e-3, 2.0, 1.5, S, S, F, out)
    v, th = [x.copy() for x in s[:3]], s[3].copy()
    og.bouss_step(v, th, 1e-3, 4e-3, 5e-3, 2.0, 1.5, f=f[:3], fs=f[3], ord=1)
    check(out, v + [th], m)
