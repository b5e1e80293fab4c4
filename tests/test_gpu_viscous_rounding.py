"""The viscous step's right-hand side is rounded as the reference's: without
viscosity the system is the identity and the step is its right-hand side, which
has to be ``oracle.dns``'s bit for bit (every product and sum in the same order;
the predicted pressure gradient included)."""
import numpy as np
import pytest

from test_gpu_flow import _axes
from test_gpu_flow_edges import _box, _handle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("var", [1, 2, 3, 5])
@pytest.mark.parametrize("n,lx", [((6, 10, 16), 1), ((10, 6, 17), 1), ((64, 3, 77), 6), ((2, 2, 255), 1)])
def test_step_without_viscosity_is_its_right_hand_side(cuda, var, n, lx):
    torch = cuda
    from anelastic_solve_amd import FlowBC
    from oracle import dns
    g = _box(n)
    s = _handle(g, lx)
    bc = FlowBC.make((True, True, False), {(3, f, var): (1, 0.3) for f in (1, 2)})
    rng = np.random.Generator(np.random.PCG64(36))
    v1, v2, p = (rng.standard_normal(g.shape) for _ in range(3))
    p = None if var == 5 else p
    args = (0.9, 0.45, 0.7, 0.02, var)
    want = dns.cn_advance(v1, v2.copy(), *args, g.rho_or_ones(), _axes(g), bc.TB, bc.VB, 0.0, 1.4, 0.9, p=p)
    d1, d2 = (torch.from_numpy(a).cuda() for a in (v1, v2))
    s.var_advance_CN_PL(d1, d2, *args, bc, 0.0, 1.4, 0.9, p=None if p is None else torch.from_numpy(p).cuda())
    got = d2.cpu().numpy()
    s.close()
    assert np.array_equal(got, want), np.abs(got - want).max()
