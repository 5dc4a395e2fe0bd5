"""A learned step that is run again after a failed short sort draws its check's samples
with the same number as before, and so do the replays after a failed one: the checks of
captured steps are those of eager steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 150001


@pytest.mark.parametrize("nsteps", [1, 3])
def test_checks_of_redone_steps(bt, nsteps):
    dt = 1.0 / 256
    pos, vel = bt.plummer(N, seed=51)
    rng = np.random.default_rng(5)
    k = rng.choice(N, 300, replace=False)   # the first drift brings them together
    shift = rng.uniform(-0.2, 0.2, (300, 3))
    pos[k, :3] = 0.71 + 1e-6 * rng.standard_normal((300, 3)) + shift
    vel[k, :3] = -shift / dt
    ts = []
    for _ in range(2):
        t = bt.Treecode(0.05, 0.6, 64)
        t.alloc(N)
        t.ptcl_h2d(pos, vel)
        t.use_learned_theta(check_samples=200, p99_max=1.0)
        t.buildTree(16)
        t.computeMultipoles()
        t.makeGroups(5, 64)
        t.computeForces()
        ts.append(t)
    eager, graph = ts
    try:
        for again in range(2):
            for _ in range(nsteps):
                eager.step(dt, 16, 5, 64)
            graph.step_graph(dt, 16, 5, 64, nsteps=nsteps)
            assert eager.opening_check() == graph.opening_check(), again
            assert np.array_equal(eager.check_samples(), graph.check_samples()), again
        assert eager.opening_check()["checks"] == 1 + 2 * nsteps
        assert np.array_equal(eager.acc(bt.ORDER_INPUT), graph.acc(bt.ORDER_INPUT))
    finally:
        eager.close()
        graph.close()
