"""The wall update's launch shapes: float64 plans split the 16-row blocks of a
z line over 4 or 8 waves with equal shares, mixed plans give each wave nine.
Every share is run at the ends of its range against the oracle, with the
tolerances of the other wall tests: 1e-12 of the largest value, 1e-10 for d = 8,
whose continuation moves the oracle itself by 1.2e-11 for one ulp of input."""
import numpy as np
import pytest

from conftest import TABLES, rel_err

pytestmark = pytest.mark.gpu

# nz with 8 | 9 .. 36 | 37 .. 72 | 73 blocks, and the ends of the shares between
EDGES = (36, 64, 65, 96, 97, 128, 160, 161, 192, 193, 224, 225, 256, 257, 288, 289, 320, 321, 577)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("d,nz", [(5, n) for n in EDGES] + [(8, n) for n in (44, 91, 155, 288, 289)])
def test_wall_update(d, nz, precision):
    import torch
    from oracle import specter_ref as O
    from specter_amd import FCPlan
    C = {5: 25, 8: 27}[d]
    shape = (6, 10, nz)  # 40 lines: two and a half tiles
    g = O.make_grid(*shape, C, d, TABLES)
    rng = np.random.default_rng(nz)
    th = rng.standard_normal(g.spec_shape) + 1j * rng.standard_normal(g.spec_shape)
    ref = th.copy()
    O.s_imposebc(g, ref)
    p = FCPlan(*shape, C, d, precision=precision)
    t = torch.as_tensor(th).cuda()
    p.s_imposebc(t)
    assert rel_err(t.cpu().numpy(), ref) < (1e-12 if d == 5 else 1e-10)
