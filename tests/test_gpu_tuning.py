"""Launch-shape overrides: they leave the results alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def lib():
    from specter_amd import lib as L
    lib = L.load_library()
    L.check(lib.spx_tune_clear())
    yield lib
    L.check(lib.spx_tune_clear())


def _run(shape, d, precision):
    """one gradre, one wall update and a diagnostic of a plan"""
    import torch
    from specter_amd import FCPlan
    nx, ny, nz = shape
    p = FCPlan(nx, ny, nz, {5: 25, 8: 27}[d], d, precision=precision)
    rng = np.random.default_rng(nz)
    s = p.empty_spectral().shape
    v = [torch.as_tensor(rng.standard_normal(s) + 1j * rng.standard_normal(s)).cuda()
         for _ in range(4)]
    out = [p.empty_nonlinear() for _ in range(3)]
    p.gradre(*v[:3], *out)
    e = p.cross(*v[:3], *v[1:])
    p.v_imposebc_and_project(*v, 1, 2)
    p.sync()
    return out + v + [torch.as_tensor(np.atleast_1d(e))]


def _same(a, b):
    import torch
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("n,d", [(32, 8), (64, 5), (64, 8), (128, 5), (192, 8)])
def test_shipped_choices_keep_the_results(lib, n, d):
    """a float64 run served with the shipped choices equals a run on its own to the bit"""
    from specter_amd import autotune
    shape = (6, 6, n + {5: 25, 8: 27}[d])
    ref = _run(shape, d, 0)
    assert autotune.apply_tuning() >= 0
    out = _run(shape, d, 0)
    assert _same(ref, out)
