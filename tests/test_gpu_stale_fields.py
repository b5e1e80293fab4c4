"""A V-cycle starts its levels from zero: what an earlier solve (one that met
NaN, say) left in their fields does not reach the next one.  Odd plane counts
behind walls are the case to watch, where a point half-sweep's coupling past a
wall is zero but its neighbour, by wrapping, a cell of the sweep's own colour.
NaN planted in every level's solution, then a solve against the oracle's (FP64
1e-8 after three cycles, mixed 1e-3: the residual's rounding noise is far
below either)."""
import numpy as np
import pytest

from conftest import oracle_levels, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,nlevels,pre,post", [
    ((64, 60, 21), (6, 3, 1), 3, 2),      # small levels: one launch per half-sweep or sweep, then the tail
    ((64, 60, 21), (6, 3, 1), 1, 1),
    ((256, 256, 33), (8, 6, 1), 1, 1),    # the finest level marches in z
])
def test_point_cycle_ignores_stale_fields(cuda, precision, n, nlevels, pre, post):
    torch = cuda
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import vcycle as VC
    nx, ny, nz = n
    tbc = (2, 2, 1, 1, 2, 2)
    g = box_grid(nx, ny, nz, beta=1.2)
    s = PressureSolver(g, default_config(precision=precision, smoother="RBPGS", tbc=tbc, vbc=[0.0] * 6,
                                         pre=pre, post=post, tol=1e-14, maxcy=3, pair_cycles=0,
                                         nlevels=nlevels))
    levs, fac = oracle_levels(g, tbc, s.levels, nlevels)
    for l, lv in enumerate(s.levels):
        s.level_field(l, 0, np.full((lv[2], lv[1], lv[0]), np.nan))
    b = np.zeros(g.shape)
    b[1:-1, 1:-1, 1:-1] = np.random.Generator(np.random.PCG64(8)).standard_normal((nz, ny, nx))
    bb = b[1:-1, 1:-1, 1:-1]
    p = torch.zeros(g.shape, dtype=torch.float64, device="cuda")
    s.mg_solver(p, torch.from_numpy(b).cuda())
    ld = s.direct_level
    s.close()
    ref, _ = VC.solve(levs, fac, list(tbc), [0.0] * 6, np.zeros_like(bb), bb, pre=pre, post=post,
                      smoother="RBPGS", mixed=precision == "mixed", tol=1e-14, maxcy=3,
                      direct_level=ld if ld >= 0 else None)
    assert relerr(p.cpu().numpy()[1:-1, 1:-1, 1:-1], ref) <= (1e-8 if precision == "fp64" else 1e-3)
