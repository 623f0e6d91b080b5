"""The diagnostics' sums are added in one order wherever that is done: on the host for
few values, by a kernel for more.  A member of a batch whose values go through the
kernel has the bits of the same fields in a plan of their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 9 * 8 = 72 lines, 17 * 32 = 544, 33 * 62 = 2046 (two values a thread), against 2048 values
@pytest.mark.parametrize("nx,ny,members", [(16, 8, 40), (32, 32, 8), (64, 62, 2)])
def test_host_and_device_sums_agree(nx, ny, members):
    import torch
    from specter_amd import FCPlan

    def values(p, t):
        v = [p.energy(*t[:3], 1), p.energy(*t[:3], 0), p.divergence(*t[:3]), p.variance(t[0], 0),
             p.product(t[0], t[1]), p.cross(*t[:3], *t[1:]), p.helicity(*t[:3]),
             *p.bouncheck_z(t[0]), *p.bouncheck_z(t[0], t[1])]
        return np.array(v, dtype=float).reshape(len(v), -1)

    rng = np.random.default_rng(nx)
    p = FCPlan(nx, ny, 41, 25, 5, members=members)
    shape = (members, nx // 2 + 1, ny, 41)
    t = [torch.as_tensor(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).cuda()
         for _ in range(4)]
    got = values(p, t)
    one = FCPlan(nx, ny, 41, 25, 5)
    for m in (0, members - 1):
        assert np.array_equal(got[:, m], values(one, [x[m].contiguous() for x in t])[:, 0])
