"""The FP64 z-line half-sweep of a launch with more 64-column groups than the
device has compute units, which takes workgroups of 32 columns with two
segments per wave: against the 64-column shape bit for bit (every lane does
the same operations in both), and against the oracle's sweep to FP64 rounding
(1e-12 relative, as the smaller launches).  The sizes hold an odd count of
groups, a last segment of two cells, an odd count of segments."""
import numpy as np
import pytest

from conftest import oracle_levels, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tbc,nlevels", [
    ((256, 144, 18), (0, 0, 0, 0, 0, 0), (8, 4, 1)),    # 2 segments, the last of 2 cells; periodic z
    ((256, 144, 36), (2, 2, 1, 1, 2, 2), (7, 5, 2)),    # 3 segments: a wave's second one is spare
    ((144, 248, 32), (1, 2, 1, 1, 2, 2), (4, 4, 6)),    # 279 groups, whole segments
])
def test_fp64_zline_paired_segments(cuda, n, tbc, nlevels):
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import vcycle as VC
    nx, ny, nz = n
    g = box_grid(nx, ny, nz, beta=1.5, rho=1.0 - 0.1 * np.linspace(-0.05, 1.05, nz + 2))
    vbc = [0.0 if t else -1.0 for t in tbc]
    s = PressureSolver(g, default_config(smoother="LJ", precision="fp64", tbc=tbc, vbc=vbc,
                                         nlevels=nlevels))
    lev = oracle_levels(g, tbc, s.levels, nlevels)[0][0]
    rng = np.random.default_rng(11)
    u = rng.standard_normal((nz, ny, nx))
    f = rng.standard_normal((nz, ny, nx))

    def run(which):
        s.level_field(0, 0, u)
        s.level_field(0, 1, f)
        s.run_kernel(which, 0, 1)
        return s.level_field(0, 0)

    for which, forced, parity in ((0, 12, 0), (4, 13, 1)):
        got = run(which)
        assert np.array_equal(got, run(forced)), which
        ref = u.copy()
        VC.zline_half_sweep(ref, f, lev, parity, np.float64)
        assert relerr(got, ref) < 1e-12, which
    got = run(6)
    ref = np.zeros_like(u)
    VC.zline_half_sweep(ref, f, lev, 0, np.float64)
    m = VC.colour_mask(u.shape, 0, True)
    assert relerr(got[m], ref[m]) < 1e-12
    s.close()
