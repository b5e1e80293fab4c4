"""The bytes that a solve reports for its V-cycles (``bytes_cycles``), with the
point smoother on two launched levels, the second solved directly: per cell of the
first, 3w for a sweep of two launches and 2.5w for one that runs in a pair (b and
half of u read, u written), 1.625w and 1.125w for the 2:2:2 transfers, whose
solved and rewritten halves are skipped; 2w per cell of the direct level; 16 or
32 bytes per cell for the FP64 residual or correction.  Exact but for the
truncation to a whole byte."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,pre,post,paired", [
    ((64, 64, 64), 2, 2, 4),
    ((64, 64, 64), 3, 2, 4),           # the third sweep by itself
    ((64, 64, 64), 1, 1, 0),           # no pair
    ((352, 32, 32), 2, 2, 0),          # rows too long for a pair
])
def test_bytes_of_point_cycles(cuda, precision, n, pre, post, paired):
    torch = cuda
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    g = box_grid(*n, beta=0.0)
    levels = (4, 4, 4) if n[0] == 64 else (5, 4, 4)
    s = PressureSolver(g, default_config(precision=precision, smoother="RBPGS", tbc=(0, 1, 0, 1, 0, 0), pre=pre,
                                         post=post, tol=1e-3, maxcy=3, pair_cycles=0, nlevels=levels))
    assert s.direct_level == 1
    rhs = torch.randn(g.shape, generator=torch.Generator(device="cuda").manual_seed(1), dtype=torch.float64,
                      device="cuda")
    it, _ = s.mg_solver(torch.zeros_like(rhs), rhs)
    got, cycles = s.stats.bytes_cycles, min(it, 3)
    s.close()
    w, cells = 8.0 if precision == "fp64" else 4.0, n[0] * n[1] * n[2]
    per = w * cells * (3.0 * (pre + post) - 0.5 * paired + 1.625 + 1.125) + 2.0 * w * cells / 8
    per += (16.0 if precision == "fp64" else 32.0) * cells
    assert got == pytest.approx(cycles * per, abs=cycles)
