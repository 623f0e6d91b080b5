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
