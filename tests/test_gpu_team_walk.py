"""Small systems are walked by teams of four waves per group: the same
interaction lists as one wave per group (blocks_per_cu set by hand keeps to
that), and forces that agree to the rounding of their sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _walks(bt, n, ncrit=64, theta=0.5, fp64=False, mono=False, learned=False, kahan=1, mode=0,
           offsets=None):
    pos, vel = bt.plummer(n, seed=31)
    t = bt.Treecode(0.01, theta, ncrit, fp64=fp64)
    t.alloc(n, offsets)
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.computeMultipoles()
    t.set_group_mode(mode)
    t.makeGroups(5, ncrit)
    if mono:
        t.set_quadrupole(False)
    if learned:
        t.use_learned_theta(check_samples=0)
    out = []
    for blocks_per_cu in (0, 8):
        t.set_walk_options(kahan=kahan, blocks_per_cu=blocks_per_cu)
        st = t.computeForces()
        out.append((t.acc(bt.ORDER_PH).astype(np.float64), t.group_counts(), st,
                    t.grav_potential, t.walk_stack_max()))
    t.close()
    return out


def _compare(team, wave, tol):
    assert np.array_equal(team[1], wave[1])          # interactions per group
    assert team[2] == wave[2]
    assert team[4] + 1024 >= wave[4]      # a stack sized by it (and the LDS part) holds either walk
    d = np.linalg.norm(team[0] - wave[0]) / np.linalg.norm(wave[0])
    assert d <= tol, d
    assert abs(team[3] - wave[3]) <= tol * abs(wave[3])


# each side sums about 2^12 terms, compensated every 64: a few 2^-24 apart
@pytest.mark.parametrize("n", [2, 3, 65, 257, 1025, 10007, 1 << 16, 1 << 19])
def test_team_walk_matches_wave_walk(bt, n):
    _compare(*_walks(bt, n), 1e-6)


@pytest.mark.parametrize("kw", [dict(kahan=0), dict(mono=True), dict(learned=True), dict(ncrit=7),
                                dict(mode=1), dict(mode=2), dict(theta=1.5)],
                         ids=lambda k: "%s=%s" % next(iter(k.items())))
def test_team_walk_options(bt, kw):
    _compare(*_walks(bt, 20011, **kw), 1e-6)


def test_team_walk_fp64(bt):
    _compare(*_walks(bt, 9001, fp64=True), 1e-13)
    _compare(*_walks(bt, 9001, fp64=True, mono=True), 1e-13)


def test_team_walk_forest(bt):
    off = np.array([0, 1, 3, 700, 701, 5000, 9001], np.int32)
    _compare(*_walks(bt, 9001, offsets=off), 1e-6)


def test_team_walk_spills(bt):
    """A tiny angle opens every node, so a step's children outgrow the 2048
    stack entries a team keeps in LDS."""
    team, wave = _walks(bt, 1 << 17, theta=0.03)
    assert team[4] > 2048
    _compare(team, wave, 1e-6)
