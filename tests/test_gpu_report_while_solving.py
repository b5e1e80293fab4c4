"""The divergence report of a handle while another thread solves with it: the
report's results have a place of their own, so both are what they are alone.
(Graphs off: a stream that is being captured takes no other launches.)"""
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_divergence_report_during_solves(cuda):
    torch = cuda
    from anelastic_solve_amd import PressureSolver, box_grid, default_config
    g = box_grid(64, 64, 64, beta=1.5)
    s = PressureSolver(g, default_config(tbc=(0, 1, 0, 1, 0, 0), tol=1e-10, use_graph=0))
    gen = torch.Generator(device="cuda").manual_seed(9)
    u, v, w, rhs = (torch.randn(g.shape, generator=gen, dtype=torch.float64, device="cuda") for _ in range(4))
    div = torch.zeros_like(u)
    p0 = torch.zeros_like(u)
    it0, _ = s.mg_solver(p0, rhs)
    want = s.divergence(u, v, w, div)
    guesses = [torch.zeros_like(u) for _ in range(40)]
    torch.cuda.synchronize()
    got, done = [], threading.Event()

    def report():
        while not done.is_set():
            got.append(s.divergence(u, v, w, div))

    t = threading.Thread(target=report)
    t.start()
    try:
        its = [s.mg_solver(p, rhs)[0] for p in guesses]
    finally:
        done.set()
        t.join()
    s.close()
    print(f"{len(got)} reports, {sum(r != want for r in got)} wrong", flush=True)
    assert len(got) > 20 and all(r == want for r in got)
    assert its == [it0] * len(its)
    assert all(torch.equal(p, p0) for p in guesses)
