"""The residual restriction of levels too small to march (four lanes per
coarse cell): in full against the oracle, and as the V-cycle runs it, with the
residuals of the cells that the pre-smoothing's last half-sweep solved taken
as zero.  Tolerances as the marching restriction's: FP64 1e-12, FP32 2e-5 of
the largest value."""
import numpy as np
import pytest

from conftest import oracle_levels, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("smoother", ["LJ", "RBPGS"])
@pytest.mark.parametrize("n,tbc", [
    ((4, 4, 4), (2, 2, 1, 1, 2, 2)),          # eight coarse cells: half a wave
    ((12, 20, 28), (0, 1, 0, 1, 0, 0)),       # 840 coarse cells: a short last block
    ((64, 48, 32), (0, 1, 0, 1, 0, 0)),       # 96 full blocks
    ((16, 12, 24), (0, 0, 0, 0, 0, 0)),       # periodic z: the z-line sweep solves nothing exactly
])
def test_restrict_quad(cuda, precision, smoother, n, tbc):
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import vcycle as VC
    nx, ny, nz = n
    levels = (4, 3, 3) if nx == 64 else (2, 2, 2)
    g = box_grid(nx, ny, nz, beta=1.5, rho=1.0 - 0.1 * np.linspace(-0.05, 1.05, nz + 2))
    s = PressureSolver(g, default_config(precision=precision, smoother=smoother, tbc=tbc,
                                         vbc=[0.0 if t else -1.0 for t in tbc], nlevels=levels))
    levs, fac = oracle_levels(g, tbc, s.levels, levels)
    assert tuple(fac[0]) == (2, 2, 2)
    dt = np.float64 if precision == "fp64" else np.float32
    rng = np.random.default_rng(3)
    u = rng.standard_normal((nz, ny, nx)).astype(dt)
    f = rng.standard_normal((nz, ny, nx)).astype(dt)
    r = VC.residual(u, f, levs[0], dt)
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    solved = ((i + j) & 1 if smoother == "LJ" else (i + j + k) & 1) == 1
    if smoother == "LJ" and tbc == (0, 0, 0, 0, 0, 0):
        solved[:] = False
    for which in (1, 16):
        s.level_field(0, 0, u)
        s.level_field(0, 1, f)
        s.run_kernel(which, 0, 1)
        if which == 16:
            r[solved] = 0
        ref = VC.restrict(r, levs[0], levs[1], fac[0], dt)
        assert relerr(s.level_field(1, 1), ref) < (1e-12 if precision == "fp64" else 2e-5), which
    s.close()
