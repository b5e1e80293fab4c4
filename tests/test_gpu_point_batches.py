"""Paired point sweeps of several instances in one launch (rows of different
widths under the widest's thread count, slabs of two and of four planes, odd and
even nz): every member's pressure is bitwise that of its solve alone."""
import pytest

pytestmark = pytest.mark.gpu

# nlevels (6, 5, 1): x and y coarsened, every level's nz that of the grid
SIZES = [(64, 128, 32),      # hx 32: 32 x 8 tiles, slabs of four
         (192, 64, 9),       # hx 96: two
         (320, 64, 21),      # hx 160: two
         (64, 160, 29),      # 40 x 8 tiles: four, odd nz
         (64, 32, 4)]        # the smallest nz a pair takes
CFG = dict(smoother="RBPGS", tbc=(0, 1, 0, 2, 0, 0), nlevels=(6, 5, 1), tol=1e-14, maxcy=4)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("pre,post", [(2, 2), (3, 1)])
def test_point_batch_equals_alone(cuda, precision, pre, post):
    torch = cuda
    from anelastic_solve_amd import BatchSolver, PressureSolver, box_grid, default_config
    cfg = dict(CFG, precision=precision, pre=pre, post=post)
    grids = [box_grid(*n, beta=0.8) for n in SIZES]
    gen = torch.Generator(device="cuda").manual_seed(12)
    rhs = [torch.randn(g.shape, generator=gen, dtype=torch.float64, device="cuda") for g in grids]
    both = []
    for g, b in zip(grids, rhs):
        s = PressureSolver(g, default_config(**cfg))
        both.append(torch.zeros_like(b))
        s.mg_solver(both[-1], b)
        s.close()
    bs = BatchSolver(grids, default_config(**cfg))
    phis = [torch.zeros_like(b) for b in rhs]
    bs.solve(phis, rhs)
    for n, p, want in zip(SIZES, phis, both):
        assert torch.isfinite(want).all() and want.abs().max() > 0
        assert torch.equal(p, want), n
