"""``Psource`` on both sides of each line between its slabs of one, two and
eight planes (1024 workgroups of one plane, 4096 of eight), with a short last
slab, to 1e-13 (a handful of roundings per cell)."""
import numpy as np
import pytest

from conftest import relerr
from test_gpu_flow import _axes
from test_gpu_flow_edges import _box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,levels", [
    ((64, 48, 45), (6, 5, 1)),         # 13 x 47 workgroups of one plane
    ((32, 64, 110), (5, 6, 2)),        # 9 x 112: still one
    ((32, 64, 120), (5, 5, 4)),        # 9 x 122: slabs of two
    ((96, 64, 65), (5, 6, 1)),         # two, the last slab one plane
    ((256, 256, 117), (8, 8, 1)),      # 261 x 15 workgroups of eight planes: still two
    ((256, 256, 119), (8, 8, 1)),      # 261 x 16: eight, one plane left over
])
def test_source_slabs(cuda, n, levels):
    torch = cuda
    from anelastic_solve_amd import PressureSolver, default_config
    from oracle import ops
    g = _box(n)
    s = PressureSolver(g, default_config(precision="fp64", smoother="RBPGS", tbc=(2,) * 6, vbc=(0.0,) * 6,
                                         nlevels=levels))
    rng = np.random.Generator(np.random.PCG64(33))
    U, V, W = (rng.standard_normal(g.shape) for _ in range(3))
    S = torch.full(g.shape, 7.0, dtype=torch.float64, device="cuda")
    s.psource(*(torch.from_numpy(a).cuda() for a in (U, V, W)), S, 0.3)
    s.close()
    assert relerr(S.cpu().numpy(), ops.psource(U, V, W, g.rho, *_axes(g), 0.3)) < 1e-13
