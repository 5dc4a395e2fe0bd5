"""A HIP error that the caller's own code left behind (an allocation that did not fit) is
not an error of the calls that set particles and read results, and stays the caller's."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_results_after_a_foreign_error(bt):
    hip = ctypes.CDLL("libamdhip64.so")
    n = 1000
    pos, vel = bt.plummer(n, seed=3)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(n)
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.computeMultipoles()
    t.makeGroups(5, 64)
    t.computeForces()
    acc = t.acc(bt.ORDER_INPUT)

    def foreign_error():
        p = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0
    foreign_error()
    assert np.array_equal(t.acc(bt.ORDER_INPUT), acc)
    p, v = t.ptcl_d2h(bt.ORDER_INPUT)
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    t.ptcl_h2d(pos, vel)
    assert hip.hipGetLastError() != 0
    t.close()
