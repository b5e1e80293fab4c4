"""The coarse tail of levels whose columns share one matrix (k_tail_line) by
itself: which solvers run it, and one sub-V-cycle of it against the oracle's in
FP64.  Its FP32 sweeps, transfers and weights carry roundings of about 1e-7 of
the largest value each, some tens of them in a value: 2e-5, as for the
restriction."""
import numpy as np
import pytest

from conftest import oracle_levels, relerr
from test_gpu_line_tail import CASES

pytestmark = pytest.mark.gpu


def _levels_of_the_tail(s):
    from anelastic_solve_amd._capi import AMGError
    found = []
    for l in range(len(s.levels)):
        try:
            s.run_kernel(18, l, 0)
            found.append(l)
        except AMGError:
            pass
    return found


@pytest.mark.parametrize("n,tbc,pre,post", CASES)
def test_line_tail_is_the_oracles_cycle(cuda, n, tbc, pre, post):
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    from oracle import ops, vcycle as VC
    g = box_grid(*n, beta=1.6)
    s = PressureSolver(g, default_config(precision="mixed", tbc=tbc, vbc=[-1.0 if t == 0 else 0.0 for t in tbc],
                                         pre=pre, post=post))
    at = _levels_of_the_tail(s)
    assert len(at) == 1
    levs, fac = (a[at[0]:] for a in oracle_levels(g, tbc, s.levels))
    nx, ny, nz = s.levels[at[0]]
    f = np.random.Generator(np.random.PCG64(43)).standard_normal((nz, ny, nx)).astype(np.float32).astype(np.float64)
    if 2 not in tbc:
        f = ops.compat_project(f, levs[0]).astype(np.float32).astype(np.float64)
    s.level_field(at[0], 1, f)
    s.run_kernel(18, at[0], 1)
    got = s.level_field(at[0], 0)
    s.close()
    minv = VC.coarse_operator_inverse(levs[-1], 2 not in tbc)
    L = len(levs)
    ref = VC.vcycle(levs, fac, np.zeros_like(f), f, [pre] * L, [post] * L, "LJ", np.float64, minv, zero_guess=True)
    err = relerr(got, ref)
    print(f"{n}: from level {at[0]}, {err:.1e}", flush=True)
    assert err <= 2e-5


@pytest.mark.parametrize("kw,tbc", [
    (dict(precision="fp64"), (0, 1, 0, 1, 0, 0)),
    (dict(precision="mixed", smoother="RBPGS"), (0, 1, 0, 1, 0, 0)),
    (dict(precision="mixed"), (0, 0, 0, 0, 0, 0)),                    # periodic z
    (dict(precision="mixed", pre=0), (0, 1, 0, 1, 0, 0)),
    (dict(precision="mixed", nlevels=(3, 3, 2)), (0, 1, 0, 1, 0, 0)),   # no 2:2:2 transfer to the last level
])
def test_other_tails(cuda, kw, tbc):
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    s = PressureSolver(box_grid(32, 24, 16, beta=1.0), default_config(tbc=tbc, vbc=[-1.0 if t == 0 else 0.0 for t in tbc], **kw))
    found = _levels_of_the_tail(s)
    s.close()
    assert found == []
