"""The adaptive tree against the oracle's, bit for bit, where the order of a leaf's
bodies comes about differently: one leaf (input order), leaves of up to 1024
bodies (a wave each) and larger ones (a sort), on one handle that changes between
them, in clustered bodies and with as many in one place as a leaf takes."""
import ctypes

import numpy as np
import pytest

import exafmm_hip as X
from helpers import plummer, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


def check(f, x, ncrit):
    f.set_bodies(x)
    f.get_bounds()
    f.build_tree()
    f.upward_pass()
    o = run_oracle(x, P=4, ncrit=ncrit, adaptive=True)
    c, oc = f.cells(), o.cells()
    for k in ("iparent", "ichild", "nchild", "ibody", "nbody", "X", "R"):
        assert np.array_equal(c[k], oc[k]), k
    b, ob = f.bodies(), o.bodies()
    assert np.array_equal(b["ibody"], ob["ibody"])
    assert np.array_equal(b["xyzq"], ob["xyzq"])


@pytest.mark.parametrize("ncrit", [1000, 1024, 1025, 3000, 4000])
def test_leaves_match_oracle(ncrit):
    print(f"[gpu] adaptive build, leaves of up to {ncrit}", flush=True)
    f = X.FMM(P=4, ncrit=ncrit, builder="adaptive")
    heap = plummer(9000, 3)
    heap[::9, :3] = heap[0, :3]
    for x in (unit_cube(6000, 1), plummer(9000, 2), unit_cube(ncrit, 4), unit_cube(ncrit + 1, 5), unit_cube(2, 6), heap,
              unit_cube(6000, 7)):
        check(f, x, ncrit)
    f.close()


def test_more_nodes_than_one_launch_takes():
    """83 M nodes: 2^26 workgroups of 64 are more than a launch takes."""
    n = 56_000_000
    x = np.random.default_rng(5).random((n, 4))
    print("[gpu] adaptive build, 83 M nodes", flush=True)
    f = X.FMM(P=4, ncrit=1, builder="adaptive")
    f.set_bodies(x)
    f.get_bounds()
    assert f.build_tree() > 1 << 26
    f.upward_pass()
    f.synchronize()
    ib = np.empty(n, np.int32)
    f._check(f.lib.exafmm_hip_get_bodies(f.h, None, ib.ctypes.data_as(ctypes.c_void_p), None), "get_bodies")
    assert (np.bincount(ib, minlength=n) == 1).all()
    f.close()
