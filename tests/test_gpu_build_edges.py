"""The cell build at the edges of its tiles and windows: cells equal to the
oracle's, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _line(bt, n):
    pos, vel = bt.plummer(n, seed=9)
    pos[:, 1:3] = 0.25          # one octant digit in two bits: deep, narrow trees
    return pos, vel


def _twins(bt, n):
    pos, vel = bt.plummer(n, seed=8)
    pos[: n // 2, :3] = pos[0, :3]      # half of them on one point: depth-capped leaf
    return pos, vel


# a cell tile holds 1024 particles, and the particle past the last closes the cells
@pytest.mark.parametrize("nleaf", [16, 24, 64])
@pytest.mark.parametrize("n,make", [(2, None), (17, None), (65, None), (1023, None), (1024, None),
                                    (1025, None), (2048, _line), (3000, _twins), (70001, None)])
def test_cells_match_oracle(bt, oracle, n, make, nleaf):
    pos, vel = make(bt, n) if make else bt.plummer(n, seed=7)
    ref = oracle.reference_pipeline(pos, nleaf, 64, 0.5, 0.01, level_split=5)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(n)
    t.ptcl_h2d(pos, vel)
    t.buildTree(nleaf)
    t.computeMultipoles()
    got = t.tree()
    counts = t.counts()
    t.close()
    assert np.array_equal(got["cells"], ref["tree"].cells)
    assert counts["nnodes"] + counts["nleaves"] == counts["ncells"] == len(got["cells"])
    leaves = got["cells"][:, 1] == 0xFFFFFFFF
    assert counts["nleaves"] == int(leaves.sum())
    assert np.array_equal(got["mono"], ref["mono"]) or np.allclose(got["mono"], ref["mono"],
                                                                   rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("sizes", [(1, 1, 1), (1023, 1, 1025, 40, 2), (16, 17, 15) * 90])
def test_forest_cells_match_single_systems(bt, oracle, sizes):
    """A forest's cells are its systems' cells, level by level and system by system."""
    parts = [bt.plummer(max(k, 2), seed=20 + i) for i, k in enumerate(sizes)]
    pos = np.concatenate([p[:k] for (p, _), k in zip(parts, sizes)])
    vel = np.concatenate([v[:k] for (_, v), k in zip(parts, sizes)])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(len(pos), off)
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.computeMultipoles()
    got = t.tree(multipoles=False)["cells"].astype(np.int64)
    t.close()
    want = []
    for b, e in zip(off[:-1], off[1:]):
        c = oracle.reference_pipeline(pos[b:e], 16, 64, 0.5, 0.01,
                                      level_split=5)["tree"].cells.astype(np.int64)
        for x, y, pb, pe in c:
            nchild = 0 if y == 0xFFFFFFFF else (y >> 29) + 1
            want.append((x >> 27, int(b) + pb, int(b) + pe, nchild))
    have = [(x >> 27, pb, pe, 0 if y == 0xFFFFFFFF else (y >> 29) + 1) for x, y, pb, pe in got]
    assert sorted(have) == sorted(want)
    for i, (x, y, pb, pe) in enumerate(got):        # links: children of i name i as their parent
        if y != 0xFFFFFFFF:
            first, nchild = y & 0x1FFFFFFF, (y >> 29) + 1
            kids = got[first:first + nchild]
            assert (kids[:, 0] & 0x07FFFFFF == i).all() and kids[:, 2].min() == pb
            assert kids[:, 3].max() == pe


def _moments(t):
    """Cells' moments by (level, particle range)."""
    g = t.tree()
    rows = {}
    for k, (x, y, pb, pe) in enumerate(g["cells"].tolist()):
        rows[(x >> 27, pb, pe)] = (g["size"][k].tobytes(), g["mono"][k].tobytes(),
                                   g["q0"][k].tobytes(), g["q1"][k].tobytes())
    return rows


@pytest.mark.parametrize("fp64", [False, True])
def test_moments_do_not_depend_on_the_launches(bt, fp64):
    """Small trees take their moments in one launch, larger ones level by level: a
    system's are the same bits alone and in a forest of more than 2^18 particles,
    and again when they are computed once more."""
    small, big = 5001, 1 << 18
    ps, vs = bt.clustered(small, 8, seed=41)
    pb, vb = bt.plummer(big, seed=42)
    real = np.float64 if fp64 else np.float32
    t = bt.Treecode(0.01, 0.5, 64, fp64=fp64)
    t.alloc(small)
    t.ptcl_h2d(ps.astype(real), vs.astype(real))
    t.buildTree(16)
    t.computeMultipoles()
    alone = _moments(t)
    t.set_params(theta=0.7)
    t.computeMultipoles()
    t.set_params(theta=0.5)
    t.computeMultipoles()
    assert _moments(t) == alone
    t.alloc(small + big, np.array([0, small, small + big], np.int32))
    t.ptcl_h2d(np.concatenate([ps, pb]).astype(real), np.concatenate([vs, vb]).astype(real))
    t.buildTree(16)
    t.computeMultipoles()
    both = _moments(t)
    t.close()
    assert {k: v for k, v in both.items() if k[2] <= small} == alone
