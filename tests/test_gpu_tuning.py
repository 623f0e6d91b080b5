"""Launch-shape overrides: what takes them, and that they leave the results alone."""
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
    """one gradre, one wall update and a diagnostic of a plan; its info"""
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
    return out + v + [torch.as_tensor(np.atleast_1d(e))], p.info()


def _same(a, b):
    import torch
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("nz,d,threads,precision",
                         [(91, 8, 16, 0)] + [(nz, 5, t, q) for nz, t in ((89, 16), (153, 64), (537, 64))
                                             for q in (0, 1)])
def test_compiled_lines_take_a_tuned_line_count(lib, nz, d, threads, precision):
    """one line a workgroup of a full wave, the plan's default, the most threads, and counts
    no workgroup can have; threads and table places belong to the plan"""
    from specter_amd import lib as L
    ref, info = _run((20, 6, nz), d, precision)
    assert info.z_wave_plan >= 0 and info.z_threads_per_line == threads
    most = 512 // threads
    for lines in {64 // threads, info.z_lines_per_block // 2, most, 2 * most, 3}:
        for cs in (16, 8):
            L.check(lib.spx_tune_line(nz, cs, lines, 2 * threads, 0))
        out, got = _run((20, 6, nz), d, precision)
        fits = lines <= most and lines & (lines - 1) == 0
        if fits and lines <= info.z_lines_per_block:
            assert got.z_lines_per_block == lines
        else:
            assert got.z_lines_per_block in ((lines,) if fits else ()) + (info.z_lines_per_block,)
        assert got.z_threads_per_line == threads
        assert _same(ref, out)


@pytest.mark.parametrize("nz,m,m_mixed", [(153, 315, 315), (94, 192, 189)])
def test_info_describes_the_transforms(nz, m, m_mixed):
    """the convolution that runs: the smallest compiled length from 2 nz - 1 on in float64,
    the engine's own in mixed plans (94 points: 192 and 189)"""
    from specter_amd import FCPlan
    p = FCPlan(6, 6, nz, 25, 5)
    assert p.z_fft_len == m and p.info().z_tables_global == 1
    assert FCPlan(6, 6, nz, 25, 5, precision=1).z_fft_len == m_mixed


@pytest.mark.parametrize("n,d", [(32, 8), (64, 5), (64, 8), (128, 5), (192, 8)])
def test_shipped_choices_keep_the_results(lib, n, d):
    """a float64 run served with the shipped choices equals a run on its own to the bit"""
    from specter_amd import autotune
    shape = (6, 6, n + {5: 25, 8: 27}[d])
    ref, _ = _run(shape, d, 0)
    assert autotune.apply_tuning() >= 0
    out, _ = _run(shape, d, 0)
    assert _same(ref, out)
