"""The fused x stage of the MHD products (compiled x lines of up to 8 points per
lane) against the separate transforms and product on the general engine, which
has the same passes: the same operations in the same order, so the steps agree
to the rounding that contraction may move, 1e-16 amplified by two stages of
projections (a few 1e-15 for d = 5): 1e-12 leaves two decades."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _run(nx, ny, nz, members):
    from specter_amd import FCPlan, Solver, SolverParams, ic
    plan = FCPlan(nx, ny, nz, 25, 5, members=members)
    sol = Solver(plan, SolverParams(solver="MHD", ord=2, dt=1e-3, nu=2e-3, mu=2e-3,
                                    b0=(0.4, -0.2, 0.3)))
    for m in range(members):
        where = {"member": m} if members > 1 else {}
        u = ic.spectrum_peaked_velocity(nx, ny, nz, 25, 5 + m)
        a = ic.spectrum_peaked_velocity(nx, ny, nz, 25, 50 + m)
        for name, arr in zip(("vx", "vy", "vz", "ax", "ay", "az"), (*u, *(0.3 * x for x in a))):
            sol.set_real_field(name, arr, **where)
    sol.step(2)
    return [sol.spectral(n) for n in ("vx", "vy", "vz", "ax", "ay", "az")]


@pytest.mark.parametrize("nx,ny,members", [(32, 10, 1), (48, 6, 2), (64, 6, 1), (120, 6, 1),
                                           (144, 6, 1), (192, 6, 1), (256, 6, 1), (512, 6, 1)])
def test_fused_products(monkeypatch, nx, ny, members):
    fused = _run(nx, ny, 41, members)
    monkeypatch.setenv("SPX_WAVE_XY", "0")
    for a, b in zip(fused, _run(nx, ny, 41, members)):
        assert rel_l2(np.asarray(a), np.asarray(b)) < 1e-12
