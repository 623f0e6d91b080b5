"""The diagnostics' sums over the lines of each member: fewer and more lines than
the summing workgroup's 1024 threads, one member and several, one to three
terms; tolerance of the other diagnostics tests (1e-12)."""
import numpy as np
import pytest

from conftest import TABLES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members", [1, 3])
@pytest.mark.parametrize("nx,ny", [(6, 4), (62, 32), (66, 34)])
def test_member_sums(nx, ny, members):
    import torch
    from oracle import specter_ref as O
    from specter_amd import FCPlan
    shape = (nx, ny, 41)
    g = O.make_grid(*shape, 25, 5, TABLES)
    rng = np.random.default_rng(nx + members)
    S = [[rng.standard_normal(g.spec_shape) + 1j * rng.standard_normal(g.spec_shape)
          for _ in range(members)] for _ in range(6)]
    p = FCPlan(*shape, 25, 5, members=members)
    t = [torch.as_tensor(np.stack(x) if members > 1 else x[0]).cuda() for x in S]
    got = {
        "energy": p.energy(*t[:3], 1), "enstrophy": p.energy(*t[:3], 0),
        "cross": p.cross(*t), "helicity": p.helicity(*t[:3]),
        "divergence": p.divergence(*t[:3]), "product": p.product(t[0], t[1]),
        "variance": p.variance(t[0], 0), "walls": p.bouncheck_z(t[0], t[1]),
        "wall": p.bouncheck_z(t[2])}
    got = {k: np.asarray(v, dtype=float).reshape(-1, members) for k, v in got.items()}
    for m in range(members):
        s = [x[m] for x in S]
        ref = {
            "energy": O.energy(g, *s[:3], 1), "enstrophy": O.energy(g, *s[:3], 0),
            "cross": O.cross(g, *s), "helicity": O.helicity(g, *s[:3]),
            "divergence": O.divergence(g, *s[:3]), "product": O.product(g, s[0], s[1]),
            "variance": O.variance(g, s[0], 0), "walls": O.bouncheck_z(g, s[0], s[1]),
            "wall": O.bouncheck_z(g, s[2])}
        # cross, helicity and product cancel: relative to the terms' size
        size = {k: O.energy(g, *s[:3], 1) for k in ("cross", "product")}
        size["helicity"] = np.sqrt(O.energy(g, *s[:3], 1) * O.energy(g, *s[:3], 0))
        for k, r in ref.items():
            r = np.atleast_1d(np.asarray(r, dtype=float))
            assert np.max(np.abs(got[k][:, m] - r)) <= 1e-12 * size.get(k, np.max(np.abs(r))), k
