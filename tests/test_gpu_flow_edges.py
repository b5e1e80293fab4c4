"""The flow steps' kernels at the sizes where their shapes end, through the C ABI.

* ``ghost`` in one pass: lines of one to five cells (where the rewritten
  interior layers would be read by the other face, the launches run one by
  one) and lines across block ends, every variable type, bit-exact against
  ``oracle.dns``;
* ``Psource`` and ``divergence``: slabs of fewer than 8 planes, a last slab of
  one, positions across block ends, to 1e-13 (a handful of roundings per cell);
* the viscous step's segments.
"""
import numpy as np
import pytest

from conftest import relerr
from test_gpu_flow import _axes, _tables

pytestmark = pytest.mark.gpu


def _box(n):
    from anelastic_solve_amd import box_grid
    z = np.linspace(-0.1, 1.1, n[2] + 2)
    return box_grid(*n, beta=1.2, rho=1.0 + 0.2 * np.cos(2.0 * z))


def _handle(g, lx=1):
    """A handle of any small grid: pressure walls on every face, x alone coarsened."""
    from anelastic_solve_amd import PressureSolver, default_config
    return PressureSolver(g, default_config(precision="fp64", smoother="RBPGS", tbc=(2,) * 6,
                                            vbc=(0.0,) * 6, nlevels=(lx, 1, 1)))


@pytest.mark.parametrize("n", [(2, 1, 1), (2, 2, 2), (4, 3, 3), (6, 5, 4), (2, 3, 130)])
def test_ghost_short_lines(cuda, n):
    torch = cuda
    from oracle import dns
    g = _box(n)
    s = _handle(g)
    rng = np.random.Generator(np.random.PCG64(31))
    for q, bc in enumerate(_tables()):
        for vtype in sorted(dns.GHOST_CLASS):
            v = rng.standard_normal(g.shape)
            want = dns.ghost(v.copy(), vtype, bc.TB, bc.VB, _axes(g))
            d = torch.from_numpy(v).cuda()
            s.ghost(d, vtype, bc)
            assert np.array_equal(d.cpu().numpy(), want), (n, q, vtype)
    s.close()


@pytest.mark.parametrize("n", [(2, 1, 1), (4, 3, 7), (6, 5, 8), (2, 43, 9), (30, 2, 17), (16, 16, 4)])
def test_source_and_divergence_edges(cuda, n):
    torch = cuda
    from oracle import ops
    g = _box(n)
    s = _handle(g)
    ax, ay, az = _axes(g)
    rng = np.random.Generator(np.random.PCG64(32))
    U, V, W = (rng.standard_normal(g.shape) for _ in range(3))
    dev = [torch.from_numpy(a).cuda() for a in (U, V, W)]
    S = torch.full(g.shape, 7.0, dtype=torch.float64, device="cuda")
    s.psource(*dev, S, 0.3)
    assert relerr(S.cpu().numpy(), ops.psource(U, V, W, g.rho, ax, ay, az, 0.3)) < 1e-13
    div = torch.zeros_like(S)
    avg, most, at = s.divergence(*dev, div)
    want, wavg, wmost, wat = ops.divergence(U, V, W, ax, ay, az)
    assert relerr(div.cpu().numpy()[1:-1, 1:-1, 1:-1], want) < 1e-13
    assert abs(avg - wavg) <= 1e-13 * wavg and abs(most - wmost) <= 1e-13 * wmost
    assert tuple(at) == wat
    s.close()


@pytest.mark.parametrize("var", [1, 2, 3, 5])
@pytest.mark.parametrize("n,lx", [((2, 2, 2), 1), ((6, 10, 16), 1), ((10, 6, 17), 1), ((64, 3, 77), 6),
                                  ((48, 5, 33), 4), ((2, 2, 255), 1)])
def test_viscous_step_edges(cuda, var, n, lx):
    """``var_advance_CN_PL`` on columns of one row per segment, of a full and a
    partial last segment, and of column counts that are no multiple of 64,
    against ``oracle.dns`` to 1e-13 (as in test_gpu_flow)."""
    torch = cuda
    from anelastic_solve_amd import FlowBC
    from oracle import dns
    g = _box(n)
    s = _handle(g, lx)
    t = {1: (1, 6), 2: (2, 1), 3: (1, 2), 5: (2, 2)}[var]
    if var == 5 and n[2] == 2:
        t = (1, 2)
    bc = FlowBC.make((True, True, False), {(3, 1, var): (t[0], 0.3), (3, 2, var): (t[1], -0.2)})
    rng = np.random.Generator(np.random.PCG64(33))
    v1, v2, p = (rng.standard_normal(g.shape) for _ in range(3))
    p = None if var == 5 else p
    args = (0.9, 0.45, 0.7, 0.02, var)
    want = dns.cn_advance(v1, v2.copy(), *args, g.rho_or_ones(), _axes(g), bc.TB, bc.VB, 1e-2, 1.4, 0.9,
                          p=p)
    d1, d2 = (torch.from_numpy(a).cuda() for a in (v1, v2))
    s.var_advance_CN_PL(d1, d2, *args, bc, 1e-2, 1.4, 0.9, p=None if p is None else torch.from_numpy(p).cuda())
    assert relerr(d2.cpu().numpy(), want) <= 1e-13
    s.close()
