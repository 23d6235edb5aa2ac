"""The diagnostics' walk over kz lines and the fused sums, at the shapes where
their splits change: lines shorter than a wave, not a power of two, one wave,
one block and longer than a block; x rows with and without the kernel that
reduces the maximum in the x inverse.  Against the oracle, shell sums within
1e-12 relative L2, totals within 1e-12 (the sums' order differs)."""
import numpy as np
import pytest

from test_gpu_parity import grids, rand_spec, rel, to_gpu

pytestmark = pytest.mark.gpu

SHAPES = [((8, 4, 2), False, (1, 1, 1)), ((16, 6, 24), False, (1, 1, 1)), ((24, 8, 64), True, (1.0, 2.0, 0.5)),
          ((12, 4, 96), False, (1, 1, 1)), ((32, 4, 256), False, (1, 1, 1)), ((48, 2, 384), True, (1.0, 1.0, 2.0))]


@pytest.mark.parametrize("shape,arb,L", SHAPES)
def test_sums_and_spectra(gpu, shape, arb, L):
    g, og = grids(shape, arb, L)
    v = [rand_spec(og, s) for s in (81, 82, 83)]
    w = [rand_spec(og, s) for s in (84, 85, 86)]
    V, W = [to_gpu(x) for x in v], [to_gpu(x) for x in w]
    e = og.energy(*v, 1)
    for kin in (0, 1, 2):
        assert g.energy(*V, kin) == pytest.approx(og.energy(*v, kin), rel=1e-12)
    assert g.helicity(*V) == pytest.approx(og.helicity(*v), rel=1e-12, abs=1e-12 * og.energy(*v, 0))
    assert g.divergence(*V) == pytest.approx(og.divergence(*v), rel=1e-12)
    for got, want in zip(g.hdcheck(*V, *W), og.hdcheck(*v, *w)):
        assert got == pytest.approx(want, rel=1e-12, abs=1e-12 * max(e, og.energy(*v, 0)))
    for kin, hel in ((1, 0), (0, 0), (1, 1), (0, 1), (2, 1)):
        got, want = g.spectrumc(*V, kin=kin, hel=hel), og.spectrumc(*v, kin=kin, hel=hel)
        if kin < 2:
            assert rel(got[0], want[0]) < 1e-12
        if hel:
            assert rel(got[1], want[1]) < 1e-12
    assert rel(g.heltrans(*V, *W), og.heltrans(*v, *w)) < 1e-12
    assert rel(g.crosspecc(*V, *W, shift=1.0), og.crosspecc(*v, *w, shift=1.0)) < 1e-12
    for name in ("specpara", "specperp"):
        for got, want in zip(getattr(g, name)(*V, kin=1, hel=1), getattr(og, name)(*v, kin=1, hel=1)):
            assert rel(np.array(got), np.array(want)) < 1e-12
    for kin in (0, 1):
        assert rel(g.entperp(*V, *W, kin=kin), og.entperp(*v, *w, kin=kin)) < 1e-12
        assert rel(g.entpara(*V, *W, kin=kin), og.entpara(*v, *w, kin=kin)) < 1e-12


@pytest.mark.parametrize("shape,arb,L", SHAPES)
def test_maximum(gpu, shape, arb, L):
    g, og = grids(shape, arb, L)
    v = [rand_spec(og, s) for s in (91, 92, 93)]
    V = [to_gpu(x) for x in v]
    for kin in (0, 1, 2):
        assert g.maxabs(*V, kin) == pytest.approx(og.maxabs(*v, kin), rel=1e-12)
