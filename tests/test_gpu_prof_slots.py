"""The pass profiler names what ran: small planes, whose x and y passes are one
launch, have slots of their own with that launch's bytes; larger ones the x and
y passes'."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,plane", [(32, True), (96, False)])
def test_transforms(gpu, n, plane):
    import torch
    from ghost_amd import _lib, fftp
    out = {}
    for d, name in ((fftp.FFTW_REAL_TO_COMPLEX, "fwd"), (fftp.FFTW_COMPLEX_TO_REAL, "inv")):
        p = fftp.fftp3d_create_plan((n, n, n), d)
        r = torch.zeros(p.rshape, dtype=torch.float64, device="cuda")
        c = torch.zeros(p.cshape, dtype=torch.complex128, device="cuda")
        _lib.prof_reset()
        _lib.prof_enable(True)
        if name == "fwd":
            fftp.fftp3d_real_to_complex(p, r, c)
        else:
            fftp.fftp3d_complex_to_real(p, c, r)
        torch.cuda.synchronize()
        _lib.prof_enable(False)
        out[name] = _lib.prof_read()
        real, spec = 8.0 * r.numel(), 16.0 * c.numel()
        bytes_of = {k: (cnt, b) for k, (cnt, ms, b) in out[name].items() if cnt}
        want = {"z" + name: (1, 2 * spec)}
        if plane:
            want["xyplane_" + name] = (1, real + spec)
        else:
            want.update({"x" + name: (1, real + spec), "ypass_" + name: (1, 2 * spec)})
        assert bytes_of == want
