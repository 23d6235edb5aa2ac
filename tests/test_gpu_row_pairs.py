"""x passes that pair a field's own rows: one field and odd counts of fields,
with odd and even numbers of rows (the last row alone), on row lengths whose
x forward pairs rows and on one (512) whose forward does not.  Against numpy's
transforms, relative L2 1e-13."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [1, 2, 3])
@pytest.mark.parametrize("shape", [(24, 5, 3), (32, 3, 5), (96, 4, 3), (192, 3, 3), (256, 3, 5), (384, 5, 2), (512, 3, 3)])
def test_transforms_of_nf_fields(gpu, shape, nf):
    import torch
    from ghost_amd import _lib, fftp
    nx, ny, nz = shape
    rng = np.random.default_rng(301)
    r = [rng.standard_normal((nz, ny, nx)) for _ in range(nf)]
    want = [np.ascontiguousarray(np.fft.rfftn(x).transpose(2, 1, 0)) for x in r]
    for d, src in ((fftp.FFTW_REAL_TO_COMPLEX, r), (fftp.FFTW_COMPLEX_TO_REAL, want)):
        plan = fftp.fftp3d_create_plan(shape, d)
        fwd = d == fftp.FFTW_REAL_TO_COMPLEX
        a = [torch.from_numpy(x).cuda() for x in src]
        b = [torch.full(plan.cshape, 7.0, dtype=torch.complex128, device="cuda") if fwd else
             torch.full(plan.rshape, 7.0, dtype=torch.float64, device="cuda") for _ in range(nf)]
        pa, _ka = _lib.ptr_array([x.data_ptr() for x in a])
        pb, _kb = _lib.ptr_array([x.data_ptr() for x in b])
        fn = gpu.ghx_r2c_many if fwd else gpu.ghx_c2r_many
        _lib.check(fn(plan._h, C.c_int(nf), pa, pb))
        torch.cuda.synchronize()
        for f in range(nf):
            ref = want[f] if fwd else r[f] * (nx * ny * nz)
            assert rel(b[f].cpu().numpy(), ref) < 1e-13, (d, f)
