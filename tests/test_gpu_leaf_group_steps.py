"""Groups of leaves (or of cells of at most NCRIT particles) in a step are those of the
step's own tree, which is built before them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("n", [3000, 30000, 150001])
@pytest.mark.parametrize("graph", [False, True])
def test_groups_of_the_steps_tree(bt, oracle, mode, n, graph):
    pos, vel = bt.clustered(n, seed=33)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(n)
    t.ptcl_h2d(pos, vel)
    t.set_group_mode(mode)
    if graph:                # its steps start from forces
        t.step(0.25, 16, 5, 64)
    for _ in range(3):       # a large step: the cells change throughout
        if graph:
            t.step_graph(0.25, 16, 5, 64, nsteps=1)
        else:
            t.step(0.25, 16, 5, 64)
        cells = t.tree(multipoles=False)["cells"]
        want = oracle.leaf_groups(cells) if mode == 1 else oracle.tree_groups(cells, 64)
        assert np.array_equal(t.groups(), want)
        assert np.isfinite(t.acc(bt.ORDER_PH)).all()
    t.close()
