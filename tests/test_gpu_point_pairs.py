"""Point sweeps whose two half-sweeps run in one launch (k_rb_pair), through
the V-cycle that uses them: after three cycles the pressure and its residual
are the oracle's.  FP64: both sides round the same sums, and a residual of
1e-3 or more of b carries at most 1e-12 of noise: 1e-8.  Mixed: every FP32
correction carries roundings of about 1e-6 of itself, against a residual that
a cycle shrinks by less than 100: 1e-3.

The sizes have rows and planes left over from blocks of 4 x 4 and 4 x 2, an
odd plane count behind walls, periodic directions whose halos wrap, the widest
row a workgroup takes (and one more, which keeps single half-sweeps), and
counts of sweeps with an odd one out."""
import numpy as np
import pytest

from conftest import oracle_levels, relerr

pytestmark = pytest.mark.gpu

PERIODIC_XY = (0, 1, 0, 1, 0, 0)
WALLS = (2, 2, 1, 1, 2, 2)
CASES = [
    # n, tbc, nlevels, pre, post
    ((64, 64, 64), PERIODIC_XY, None, 2, 2),
    ((64, 32, 36), (0, 0, 0, 0, 0, 0), (5, 4, 2), 2, 2),    # z periodic
    ((64, 42, 34), WALLS, (6, 2, 2), 2, 2),                 # two rows and two planes left over
    ((64, 60, 21), WALLS, (6, 3, 1), 3, 2),                 # odd nz; a single sweep after the pair
    ((48, 72, 56), PERIODIC_XY, (4, 3, 4), 1, 4),           # no pair before, two after
    ((128, 64, 38), WALLS, (6, 4, 2), 2, 2),                # the residual's slabs of 4 planes, 2 left over
    ((336, 32, 40), WALLS, (4, 4, 4), 2, 3),                # hx = 168
    ((352, 32, 40), WALLS, (5, 4, 4), 2, 2),                # hx = 176: the finest level unpaired
]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,tbc,nlevels,pre,post", CASES)
def test_point_cycles_follow_the_oracle(cuda, precision, n, tbc, nlevels, pre, post):
    torch = cuda
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import ops, vcycle as VC
    nx, ny, nz = n
    g = box_grid(nx, ny, nz, beta=1.2, rho=1.0 - 0.1 * np.linspace(-0.05, 1.05, nz + 2))
    kw = {} if nlevels is None else {"nlevels": nlevels}
    s = PressureSolver(g, default_config(precision=precision, smoother="RBPGS", tbc=tbc,
                                         vbc=[-1.0 if t == 0 else 0.0 for t in tbc], pre=pre, post=post,
                                         tol=1e-14, maxcy=3, pair_cycles=0, **kw))
    levs, fac = oracle_levels(g, tbc, s.levels, nlevels)
    b = np.zeros(g.shape)
    b[1:-1, 1:-1, 1:-1] = np.random.Generator(np.random.PCG64(8)).standard_normal((nz, ny, nx))
    bb = b[1:-1, 1:-1, 1:-1]
    if 2 not in tbc:
        bb = ops.compat_project(bb, levs[0])
    p = torch.zeros(g.shape, dtype=torch.float64, device="cuda")
    s.mg_solver(p, torch.from_numpy(b).cuda())
    rr, ld = s.stats.relres, s.direct_level
    s.close()
    ref, info = VC.solve(levs, fac, list(tbc), [0.0] * 6, np.zeros_like(bb), bb, pre=pre, post=post,
                         smoother="RBPGS", mixed=precision == "mixed", tol=1e-14, maxcy=3,
                         direct_level=ld if ld >= 0 else None)
    lim = 1e-8 if precision == "fp64" else 1e-3
    err, dr = relerr(p.cpu().numpy()[1:-1, 1:-1, 1:-1], ref), abs(rr / info["residual"][-1] - 1)
    print(f"{n} {precision}: pressure {err:.1e}, residual {rr:.3e} ({dr:.1e})", flush=True)
    assert err <= lim and dr <= lim
