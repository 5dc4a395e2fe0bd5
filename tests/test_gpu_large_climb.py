"""Trees of up to 2^20 particles take their moments in one launch, larger ones level by
level: a system's are the same bits alone and in a forest past that size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rest", [(1 << 20) - 20001, 1 << 20])
def test_same_moments(bt, rest):
    small = 20001
    ps, vs = bt.clustered(small, 8, seed=43)
    pb, vb = bt.plummer(rest, seed=44)
    t = bt.Treecode(0.01, 0.5, 64)
    rows = []
    for pos, vel, off in ((ps, vs, [0, small]),
                          (np.concatenate([ps, pb]), np.concatenate([vs, vb]),
                           [0, small, small + rest])):
        t.alloc(len(pos), np.array(off, np.int32))
        t.ptcl_h2d(pos, vel)
        t.buildTree(16)
        t.computeMultipoles()
        g = t.tree()
        cells = g["cells"]
        mine = cells[:, 3] <= small
        key = np.lexsort((cells[mine, 2], cells[mine, 0] >> 27))
        rows.append([cells[mine, 2:][key]] +
                    [g[k][mine][key] for k in ("size", "mono", "q0", "q1")])
    t.close()
    for a, b in zip(*rows):
        assert np.array_equal(a, b)
