"""The bench's bytes of the build phases are those of the kernels that run: 5 radix passes
per sort above 2^17 keys, 8 after a run of more than 256 equal leading digits, none in
tiles; per cell what the level and multipole kernels read and write."""
import types

import numpy as np
import pytest


class _Context:
    def __init__(self, keys, ncells, nnodes, ngroups):
        self.keys = np.sort(keys.astype(np.uint64))
        self.c = dict(ncells=ncells, nnodes=nnodes, ngroups=ngroups)

    def ph(self):
        return self.keys, None

    def counts(self):
        return self.c


@pytest.mark.parametrize("n,run,passes", [(1 << 17, 1, None), ((1 << 17) + 1, 1, 5),
                                          (200000, 256, 5), (200000, 257, 8)])
def test_bytes(n, run, passes):
    import bench
    keys = np.arange(n, dtype=np.uint64) << np.uint64(40)
    keys[100:100 + run] = keys[100] + np.arange(run, dtype=np.uint64)
    t = _Context(keys, 1000, 300, 70)
    bt = types.SimpleNamespace(SORT_PASSES=5)
    b = bench.hbm_phases(bt, t, dict(sort=1.0, levels=2.0), n)
    assert b["sort_passes"] == passes
    assert b["sort"]["bytes"] == (None if passes is None else 32.0 * n * passes)
    assert b["sort"]["frac"] == (None if passes is None else
                                 pytest.approx(32.0 * n * passes / 1e-3 / 8e12))
    places = 16 if passes == 5 else 0
    assert b["levels"]["bytes"] == (92 + places) * n + 76 * 1000 + 12 * 300
    assert b["levels"]["GB_s"] == pytest.approx(b["levels"]["bytes"] / 2e-3 / 1e9)
    assert b["multipoles"]["bytes"] == 16 * n + 288 * 1000
    assert b["groups"]["bytes"] == (60 + (20 if places else 0)) * n + 12 * 70
