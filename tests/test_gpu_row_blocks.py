"""The x passes of 3 * 2^k rows in 256-lane blocks: grids just beyond the 2304
wavefronts up to which rows go out one wavefront per block, so that every mixed
row length runs both (test_gpu_mixed_lines and test_gpu_row_pairs stay below).
Cross products, dot products, the tracers' inverse and the extrema in a step of
each solver, and the transforms of one field, with their bounds."""
import pytest

import test_gpu_mixed_lines as steps
import test_gpu_row_pairs as pairs

pytestmark = pytest.mark.gpu

SHAPES = [(24, 192, 256), (48, 96, 256), (96, 96, 128), (192, 48, 128)]


@pytest.mark.parametrize("shape", SHAPES)
def test_hd(gpu, shape):
    steps.test_hd(gpu, shape)


@pytest.mark.parametrize("shape", SHAPES)
def test_bouss(gpu, shape):
    steps.test_bouss(gpu, shape)


@pytest.mark.parametrize("nf", [1, 3])
@pytest.mark.parametrize("shape", SHAPES)
def test_transforms(gpu, shape, nf):
    pairs.test_transforms_of_nf_fields(gpu, shape, nf)
