"""The walk's totals are reduced by one block up to 2^17 particles and by many above:
the potential against the sum over the particles, the counts against each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [63, 131072, 131073])
def test_totals(bt, n):
    pos, vel = bt.plummer(n, seed=91)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(n)
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.computeMultipoles()
    t.makeGroups(5, 64)
    mean_direct, max_direct, mean_approx, max_approx = t.computeForces()
    pot, phi = t.grav_potential, t.acc()[:, 3].astype(np.float64)
    _, total = t.walk_stats()
    again = t.computeForces()
    pot_again = t.grav_potential
    t.close()
    assert (pos[:, 3] == pos[0, 3]).all()
    want = 0.5 * float(pos[0, 3]) * phi.sum()
    assert abs(pot - want) <= 1e-6 * abs(want)     # phi is stored in FP32
    assert total[0] == pytest.approx(mean_direct * n, rel=1e-12)
    assert total[1] == pytest.approx(mean_approx * n, rel=1e-12)
    assert mean_direct <= max_direct <= n and mean_approx <= max_approx
    assert again == (mean_direct, max_direct, mean_approx, max_approx) and pot_again == pot
