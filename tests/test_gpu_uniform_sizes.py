"""The uniform tree where its build is sized by what is possible: trees of more
than 2^26 possible leaves (depth 9, a workgroup for each would be more than a
launch takes) and of more than 2^21 possible cells, and leaves of more than 1024
bodies or trees of more than 2^20, whose order comes from a sort.  Against the same tree made here from the
bodies' Morton keys: body order, cells per level, their keys and body ranges,
all to the bit."""
import ctypes

import numpy as np
import pytest

import exafmm_hip as X
from helpers import unit_cube

pytestmark = pytest.mark.gpu


def leaf_keys(x, ncrit):
    """Depth and Morton keys on the grid that the bounds and ncrit give."""
    n = x.shape[0]
    L = 1 + int(np.log(float(n // ncrit)) / np.log(2.0) / 3) if n >= ncrit else 0
    lo, hi = x[:, :3].min(0), x[:, :3].max(0)
    mid = (lo + hi) / 2
    d = np.float64(np.float32(2 * (max((mid - lo).max(), (hi - mid).max()) * 1.00001) / 2 ** L))
    key = np.zeros(n, np.int64)
    for k in range(3):
        i = ((x[:, k] - lo[k]) / d).astype(np.int64)
        for b in range(L):
            key |= ((i >> b) & 1) << (3 * b + k)
    return L, key


def check_tree(f, x, ncrit):
    f.set_bodies(x)
    f.get_bounds()
    nc = f.build_tree()
    L, key = leaf_keys(x, ncrit)
    order = np.argsort(key, kind="stable").astype(np.int32)
    ib = np.empty(f.n, np.int32)
    f._check(f.lib.exafmm_hip_get_bodies(f.h, None, ib.ctypes.data_as(ctypes.c_void_p), None), "get_bodies")
    assert np.array_equal(ib, order)
    ints, icell = np.empty((nc, 5), np.int32), np.empty(nc, np.uint64)
    f._check(f.lib.exafmm_hip_get_cells(f.h, ints.ctypes.data_as(ctypes.c_void_p),
                                        icell.ctypes.data_as(ctypes.c_void_p), None, None, None, None), "get_cells")
    key = key[order]
    first = 0
    for t in range(L + 1):
        k = key >> (3 * (L - t))
        head = np.flatnonzero(np.concatenate([[True], k[1:] != k[:-1]]))
        m = head.shape[0]
        assert np.array_equal(icell[first:first + m], k[head][::-1].astype(np.uint64)), t
        assert np.array_equal(ints[first:first + m, 3], head[::-1]), t
        assert np.array_equal(ints[first:first + m, 4], np.diff(np.append(head, f.n))[::-1]), t
        first += m
    assert first == nc


def on_sphere(n, seed):
    x = np.random.default_rng(seed).standard_normal((n, 4))
    x[:, :3] /= np.linalg.norm(x[:, :3], axis=1)[:, None]
    return x


def corner(n, m, seed):
    """m of n bodies in one leaf."""
    x = unit_cube(n, seed)
    x[:m, :3] = 0.9 + 1e-3 * x[:m, :3]
    return x[np.random.default_rng(seed).permutation(n)]


def test_depth_nine():
    x = on_sphere((1 << 24) + 1001, 9)
    print("[gpu] uniform build, 2^27 possible leaves", flush=True)
    f = X.FMM(P=4, ncrit=1)
    check_tree(f, x, 1)
    f.close()


def test_more_cells_than_are_sized_unread():
    x = unit_cube(300000, 3)
    print("[gpu] uniform build, 2.4 M possible cells", flush=True)
    f = X.FMM(P=4, ncrit=1)
    check_tree(f, x, 1)
    check_tree(f, unit_cube(1000, 4), 1)
    check_tree(f, x, 1)
    f.close()


def test_large_leaves():
    f = X.FMM(P=4, ncrit=64)
    # Rank or sort, each after either; 1024 and 1025 bodies in a leaf of their own.
    for n, m in ((20000, 15000), (20000, 0), (70000, 66000), (70000, 60000), (3000, 0)):
        print(f"[gpu] uniform build, {m} of {n} in one leaf", flush=True)
        check_tree(f, corner(n, m, n + m), 64)
    f.close()
    for n in (1024, 1025, 1 << 20, (1 << 20) + 1):
        f = X.FMM(P=4, ncrit=1200)
        check_tree(f, unit_cube(n, n), 1200)
        check_tree(f, unit_cube(n, n + 1), 1200)
        f.close()


def test_large_leaf_in_a_forest():
    xs = [unit_cube(700, 1), corner(9000, 8000, 2), unit_cube(1, 3), corner(6000, 5000, 4)]
    print("[gpu] forest with large leaves", flush=True)
    f = X.FMM(P=4, ncrit=64)
    got = f.evaluate_batch(xs)
    ib = f.bodies()["ibody"]
    off = 0
    for x in xs:
        key = leaf_keys(x, 64)[1]
        n = x.shape[0]
        assert np.array_equal(ib[off:off + n] - off, np.argsort(key, kind="stable"))
        off += n
    assert all(np.isfinite(g[0]).all() for g in got)
    f.close()
