"""The x stages of the nonlinear term: which kernels a plan's x lines run, and
their results where a launch has one workgroup per tile instead of one per field."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _kernels(plan, call):
    """names of the kernels that call launches on the plan's stream"""
    from specter_amd import lib as L
    lib = L.load_library()
    L.check(lib.spx_prof_enable(plan.handle, 1))
    call()
    n = ctypes.c_int()
    L.check(lib.spx_prof_resolve(plan.handle, ctypes.byref(n)))
    names, launches = set(), ctypes.c_long()
    ms, nbytes = ctypes.c_double(), ctypes.c_double()
    for i in range(n.value):
        name = ctypes.create_string_buffer(64)
        L.check(lib.spx_prof_get(plan.handle, i, name, 64, ctypes.byref(launches),
                                 ctypes.byref(ms), ctypes.byref(nbytes)))
        names.add(name.value.decode())
    L.check(lib.spx_prof_enable(plan.handle, 0))
    return names


def _random(p, n, seed):
    import torch
    rng = np.random.default_rng(seed)
    shape = p.empty_spectral().shape
    return [torch.as_tensor(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).cuda()
            for _ in range(n)]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nx", [256, 512, 1024])
def test_long_x_lines_are_fused(nx, precision):
    """the whole x stage of gradre in one kernel: no real velocity goes to memory"""
    from specter_amd import FCPlan
    p = FCPlan(nx, 6, 41, 25, 5, precision=precision)
    v, out = _random(p, 3, nx), [p.empty_nonlinear() for _ in range(3)]
    names = _kernels(p, lambda: p.gradre(*v, *out))
    assert "xgrad_fused" in names and not names & {"xc2r", "xgrad_prod"}


# A launch of at least 512 tiles of the plan's own lines per workgroup runs all
# fields in one workgroup, one after the other, over the y derivatives' buffers;
# smaller ones halve the lines and give each field a workgroup.
@pytest.mark.parametrize("precision,tol", [(0, 1e-12), (1, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,npz", [(32, 256, 128), (72, 256, 128), (16, 256, 128), (512, 64, 64)])
def test_large_launches_against_the_oracle(nx, ny, npz, precision, tol):
    """gradre with full workgroups (tolerances of the other gradre tests: largest value in
    float64, L2 norm in mixed plans); 16 points run on the general engine"""
    import torch
    from conftest import TABLES, rel_err, rel_l2
    from oracle import specter_ref as O
    from specter_amd import FCPlan
    g = O.make_grid(nx, ny, npz + 25, 25, 5, TABLES)
    rng = np.random.default_rng(nx)
    v = [rng.standard_normal(g.spec_shape) + 1j * rng.standard_normal(g.spec_shape)
         for _ in range(3)]
    p = FCPlan(nx, ny, npz + 25, 25, 5, precision=precision)
    out = [p.empty_nonlinear() for _ in range(3)]
    p.gradre(*(torch.as_tensor(a).cuda() for a in v), *out)
    for o, r in zip(out, O.gradre(g, *v)):
        o = o.cpu().numpy().astype(complex)
        assert (rel_err if precision == 0 else rel_l2)(o, r) < tol


def _steps(solver, nx, ny, precision, seeds):
    """two RK2 steps of a batch with one member per seed"""
    from specter_amd import FCPlan, Solver, SolverParams, ic
    plan = FCPlan(nx, ny, 64 + 25, 25, 5, precision=precision, members=len(seeds))
    prm = dict(solver=solver, ord=2, dt=1e-3, nu=2e-3)
    if solver == "BOUSS":
        prm.update(kappa=2e-3, xmom=1.0, xtemp=1.0)
    sol = Solver(plan, SolverParams(**prm))
    names = ("vx", "vy", "vz", "th")[:3 + (solver == "BOUSS")]
    where = [{"member": m} if len(seeds) > 1 else {} for m in range(len(seeds))]
    for w, s in zip(where, seeds):
        u = list(ic.spectrum_peaked_velocity(nx, ny, 64 + 25, 25, s))
        for name, a in zip(names, u + [0.1 * u[2]]):
            sol.set_real_field(name, a, **w)
    sol.step(2)
    return [[sol.spectral(n, **w) for n in names + ("pr",)] for w in where]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("solver", ["HD", "BOUSS"])
@pytest.mark.parametrize("nx,ny", [(32, 32), (48, 32), (512, 8)])
def test_large_and_small_launches_agree(nx, ny, solver, precision):
    """16 members fill the launches, one alone does not: three fields and the scalar as
    fourth, the same bits either way"""
    seeds = list(range(40, 56))
    batch = _steps(solver, nx, ny, precision, seeds)
    for m in (0, 15):
        for a, b in zip(batch[m], _steps(solver, nx, ny, precision, seeds[m:m + 1])[0]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,fused", [(32, True), (48, True), (120, True), (144, False),
                                      (150, False), (256, True), (512, True), (1024, False)])
def test_mhd_products_are_fused(nx, fused):
    """the x stage of the cross products in one kernel for compiled x lines of up to 8
    points per lane; 144 (9), 1024 and 150 points (the engine) run separate kernels"""
    from specter_amd import FCPlan, Solver, SolverParams, ic
    plan = FCPlan(nx, 6, 41, 25, 5)
    sol = Solver(plan, SolverParams(solver="MHD", ord=2, dt=1e-4, nu=2e-3, mu=2e-3,
                                    b0=(0.4, -0.2, 0.3)))
    u = ic.spectrum_peaked_velocity(nx, 6, 41, 25, 5)
    for name, a in zip(("vx", "vy", "vz", "ax", "ay", "az"), (*u, *(0.3 * x for x in u))):
        sol.set_real_field(name, a)
    names = _kernels(plan, lambda: sol.step(1))
    assert ("xcross" in names) == fused and ("xc2r" in names) != fused
