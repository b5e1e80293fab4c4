"""The separable direct solve of a coarse level at the edges of its operand
loads: more than one 64-wide chunk of x or y per product, more column tiles
than waves, a short last chunk, a z extent that is not a multiple of 16 --
against the oracle's separable solve, with the tolerances of its other levels
(FP64 1e-11, FP32 2e-5)."""
import numpy as np
import pytest

from conftest import oracle_levels, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,tbc,nlevels,direct", [
    ((256, 32, 64), (0, 1, 0, 1, 0, 0), (6, 4, 5), (128, 16, 32)),    # two tiles per wave, two chunks of x
    ((32, 192, 34), (2, 2, 1, 1, 2, 2), (4, 6, 2), (16, 96, 17)),     # one tile, chunks of 64 + 32 in y
    ((160, 64, 42), (1, 1, 1, 1, 1, 1), (5, 5, 2), (80, 32, 21)),     # five tiles, chunks of 64 + 16 in x
])
def test_direct_level_edges(cuda, precision, n, tbc, nlevels, direct):
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import ops, vcycle as VC
    from oracle.grid import is_singular
    nx, ny, nz = n
    g = box_grid(nx, ny, nz, beta=1.5, rho=1.0 - 0.1 * np.linspace(-0.05, 1.05, nz + 2))
    vbc = [0.0 if t else -1.0 for t in tbc]
    s = PressureSolver(g, default_config(smoother="LJ", precision=precision, tbc=tbc, vbc=vbc,
                                         nlevels=nlevels))
    ld = s.direct_level
    assert ld >= 1 and s.levels[ld] == direct, (ld, s.levels)
    lev = oracle_levels(g, tbc, s.levels, nlevels)[0][ld]
    f = np.random.default_rng(5).standard_normal(tuple(reversed(lev["n"])))
    sing = is_singular(tbc)
    if sing:
        f = ops.compat_project(f, lev)
    s.level_field(ld, 1, f)
    ref = VC.separable_solve(lev, s.level_field(ld, 1), sing)   # f as stored (FP32 in mixed)
    s.run_kernel(14, ld, 1)
    err = relerr(s.level_field(ld, 0), ref)
    assert err <= (1e-11 if precision == "fp64" else 2e-5), err
    s.close()
