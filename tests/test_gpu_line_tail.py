"""The coarse tail of levels whose columns share one matrix (k_tail_line),
through the C ABI: a mixed solve on grids that such a tail cycles from the
second level (or the first) down follows the oracle's solve with the same
V-cycle -- as many cycles, the same final residual but for FP32 rounding --
and reaches the exact solution to the pressure bar of 1e-9.

An FP32 correction carries roundings of about 1e-6 of itself; a cycle
contracts by 20 or more, so a residual differs by about 1e-6 * 20 of itself
per cycle: 5e-2 leaves three decades.
"""
import numpy as np
import pytest

from conftest import oracle_levels, relerr

pytestmark = pytest.mark.gpu

CASES = [
    # n, tbc (X2max, X3min, X2min, X3max, X1min, X1max), pre, post
    ((64, 48, 32), (0, 1, 0, 1, 0, 0), 2, 2),       # 32x24x16 .. 8x6x4: 192 coarsest cells
    ((48, 48, 48), (0, 2, 0, 2, 0, 0), 2, 2),       # columns of 24 and 12 rows
    ((32, 40, 56), (0, 1, 0, 2, 0, 0), 1, 2),       # 28, 14 and 7 rows, odd y on the coarsest
    ((80, 56, 40), (0, 1, 0, 1, 0, 0), 2, 1),       # 350 coarsest cells, 5 rows
    ((16, 16, 8), (2, 2, 2, 1, 2, 2), 3, 1),        # walls in every direction, two levels
    ((32, 24, 12), (0, 1, 0, 1, 0, 0), 2, 2),       # 12, 6 and 3 rows
]


@pytest.mark.parametrize("n,tbc,pre,post", CASES)
def test_line_tail_follows_the_oracle(cuda, n, tbc, pre, post):
    torch = cuda
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import direct, ops, vcycle as VC
    nx, ny, nz = n
    g = box_grid(nx, ny, nz, beta=1.6)
    s = PressureSolver(g, default_config(precision="mixed", tbc=tbc, vbc=[-1.0 if t == 0 else 0.0 for t in tbc],
                                         pre=pre, post=post, tol=1e-11, pair_cycles=0))
    assert s.direct_level < 0
    levs, fac = oracle_levels(g, tbc, s.levels)
    b = np.zeros(g.shape)
    b[1:-1, 1:-1, 1:-1] = np.random.Generator(np.random.PCG64(42)).standard_normal((nz, ny, nx))
    bb = b[1:-1, 1:-1, 1:-1]
    if 2 not in tbc:
        bb = ops.compat_project(bb, levs[0])
    p = torch.zeros(g.shape, dtype=torch.float64, device="cuda")
    it, _ = s.mg_solver(p, torch.from_numpy(b).cuda())
    rr, ok = s.stats.relres, s.stats.converged
    s.close()
    err = relerr(p.cpu().numpy()[1:-1, 1:-1, 1:-1], direct.solve(levs[0], bb, list(tbc)))
    _, info = VC.solve(levs, fac, list(tbc), [0.0] * 6, np.zeros_like(bb), bb, pre=pre, post=post,
                       smoother="LJ", mixed=True, tol=1e-11, maxcy=100)
    print(f"{n}: {it} cycles, relres {rr:.3e}, err {err:.1e}; oracle {info['iters']}, {info['residual'][-1]:.3e}",
          flush=True)
    assert ok and err <= 1e-9
    assert it == info["iters"] and abs(rr - info["residual"][-1]) <= 5e-2 * rr
