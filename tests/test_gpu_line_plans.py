"""The compiled line plans at the edges of their ranges.

Direct plans serve z lines (of even length: x and y lines too) of exactly their
length, Rader plans z lines of M + 1, and a ladder of Bluestein lengths M every other z length with a prime
factor above 13 up to n = (M + 1) / 2: each rung is run at the smallest and the
largest n it serves.  Tolerances as for the other transform and gradre tests:
1e-13 of the largest value in float64 (the transforms), 1e-12 (gradre, d = 5),
1e-5 relative L2 for the float32 nonlinear term.  Mixed plans keep the general
engine's results to the bit: their float32 rounding decides the last digits of
the pressure."""
import numpy as np
import pytest

from conftest import TABLES, rel_err, rel_l2

pytestmark = pytest.mark.gpu

DIRECT = (24, 32, 40, 48, 60, 64, 72, 80, 88, 90, 96, 100, 108, 120, 128, 144, 160, 180, 192, 200,
          240, 256, 288, 320, 384, 512, 1024)
ODD = (75, 91, 105, 121, 125, 169, 175, 225)
RUNGS = (120, 128, 192, 256, 315, 320, 375, 384, 441, 448, 512, 640, 700, 720, 840, 900, 1080)


def _smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def _bluestein(n):
    prime = n > 1 and all(n % q for q in range(2, int(n ** 0.5) + 1))
    return not _smooth(n) and not (prime and _smooth(n - 1))


def _edges():
    out, low = [], 0
    for m in RUNGS:
        served = [n for n in range(low + 1, (m + 1) // 2 + 1) if _bluestein(n)]
        out += sorted({served[0], served[-1]})
        low = (m + 1) // 2
    return out


def _transforms(shape):
    """r2c and c2r of a periodic plan against numpy"""
    import torch
    from specter_amd import FCPlan
    nx, ny, nz = shape
    p = FCPlan(nx, ny, nz, 0, 0)
    rng = np.random.default_rng(nx + 7 * ny + 31 * nz)
    R = rng.standard_normal((nz, ny, nx))
    S = p.empty_spectral()
    p.fftp3d_real_to_complex(torch.as_tensor(R).cuda(), S)
    ref = np.fft.rfftn(R, axes=(0, 1, 2)).transpose(2, 1, 0)
    assert rel_err(S.cpu().numpy(), ref) < 1e-13
    back = p.empty_real()
    p.fftp3d_complex_to_real(torch.as_tensor(np.ascontiguousarray(ref)).cuda(), back)
    assert rel_err(back.cpu().numpy(), R * R.size) < 1e-13
    return p.info()


def _gradre(shape):
    """gradre in both precisions against the oracle"""
    import torch
    from oracle import specter_ref as O
    from specter_amd import FCPlan
    nx, ny, nz = shape
    g = O.make_grid(nx, ny, nz, 25, 5, TABLES)
    rng = np.random.default_rng(nz)
    v = [rng.standard_normal(g.spec_shape) + 1j * rng.standard_normal(g.spec_shape)
         for _ in range(3)]
    ref = O.gradre(g, *v)
    for prec in (0, 1):
        p = FCPlan(nx, ny, nz, 25, 5, precision=prec)
        out = [p.empty_nonlinear() for _ in range(3)]
        p.gradre(*(torch.as_tensor(a).cuda() for a in v), *out)
        for o, r in zip(out, ref):
            o = o.cpu().numpy().astype(complex)
            if prec == 0:
                assert rel_err(o, r) < 1e-12
            else:
                assert rel_l2(o, r) < 1e-5


def _nonlinear(shape):
    """gradre and advect of a mixed plan"""
    import torch
    from specter_amd import FCPlan
    nx, ny, nz = shape
    p = FCPlan(nx, ny, nz, 25, 5, precision=1)
    rng = np.random.default_rng(nx + 7 * ny + 31 * nz)
    v = [torch.as_tensor(rng.standard_normal(c) + 1j * rng.standard_normal(c)).cuda()
         for c in [(nx // 2 + 1, ny, nz)] * 4]
    out = [p.empty_nonlinear() for _ in range(4)]
    p.gradre(*v[:3], *out[:3])
    p.advect(*v, out[3])
    p.sync()
    return out


def _same_as_engine(monkeypatch, shape, switch):
    import torch
    compiled = _nonlinear(shape)
    monkeypatch.setenv(switch, "0")
    for a, b in zip(compiled, _nonlinear(shape)):
        assert torch.equal(a, b)
    monkeypatch.delenv(switch)


@pytest.mark.parametrize("n", _edges() + [89, 281, *ODD])
def test_z_lines(n):
    info = _transforms((6, 10, n))
    assert info.z_wave_plan >= 0
    if n >= 31:
        _gradre((6, 10, n))


@pytest.mark.parametrize("n", DIRECT)
def test_direct_lines(n):
    _transforms((n, 6, 5))
    _transforms((6, n, 5))
    if n <= 384:
        assert _transforms((6, 10, n)).z_wave_plan >= 0
    _gradre((n, 6, 41))
    _gradre((6, n, 41))


@pytest.mark.parametrize("n", [n for n in DIRECT if n != 512] + [*ODD, 57, 59, 89, 153, 217, 281, 409])
def test_mixed_plans_keep_the_bits(monkeypatch, n):
    """compiled lines against the general engine (512 and 537 have passes of
    their own)"""
    if n in DIRECT:
        _same_as_engine(monkeypatch, (n, 6, 40), "SPX_WAVE_XY")
        _same_as_engine(monkeypatch, (6, n, 40), "SPX_WAVE_XY")
    if 32 <= n <= 409:
        _same_as_engine(monkeypatch, (6, 6, n), "SPX_WAVE")
