"""The uniform tree against the oracle's, bit for bit, where the build changes
method: one leaf, prefix sums in one workgroup and in several, leaves of up to
64, 1024 and more bodies (the sort of a leaf's indices), coincident bodies,
bodies on the cell faces, and a handle whose last tree was larger or smaller.
A forest, whose systems differ in depth and share the sums, against each
system's own evaluation."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import plummer, rel_l2, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


def check(f, x, ncrit):
    f.set_bodies(x)
    f.evaluate()
    o = run_oracle(x, P=4, ncrit=ncrit)
    c, oc = f.cells(), o.cells()
    for k in ("iparent", "ichild", "nchild", "ibody", "nbody", "icell", "X", "R"):
        assert np.array_equal(c[k], oc[k]), k
    b, ob = f.bodies(), o.bodies()
    assert np.array_equal(b["ibody"], ob["ibody"])
    assert np.array_equal(b["xyzq"], ob["xyzq"])


def with_coincident(n, m):
    x = unit_cube(n, n)
    x[:m, :3] = x[0, :3]
    return x[np.random.default_rng(1).permutation(n)]


def on_faces(n):
    rng = np.random.default_rng(n)
    x = rng.integers(-8, 9, (n, 3)) / 8.0
    return np.concatenate([x, rng.uniform(-1, 1, (n, 1))], axis=1)


@pytest.mark.parametrize("name,x,ncrit", [
    ("one body", unit_cube(1, 1), 64), ("one leaf", unit_cube(63, 1), 64), ("large leaf", unit_cube(3000, 1), 4000),
    ("two levels", unit_cube(64, 2), 64), ("small", unit_cube(5000, 3), 30), ("large leaves", unit_cube(9000, 4), 4500),
    ("clustered", plummer(6000, 5), 20), ("several workgroups", unit_cube(9000, 6), 2),
    ("coincident", with_coincident(3000, 1500), 50), ("faces", on_faces(4000), 40)])
def test_tree_matches_oracle(name, x, ncrit):
    print(f"[gpu] uniform build: {name}", flush=True)
    f = X.FMM(P=4, ncrit=ncrit)
    check(f, x, ncrit)
    check(f, x, ncrit)
    f.close()


def test_larger_and_smaller_trees_on_one_handle():
    f = X.FMM(P=4, ncrit=8)
    for n in (40000, 100, 4000, 60000, 7):
        check(f, unit_cube(n, n), 8)
    f.close()


@pytest.mark.parametrize("sizes", [(1, 5000, 63, 64, 20000, 1, 700), (1,) * 300, (40000, 7, 41000)])
def test_forest_matches_single_systems(sizes):
    f = X.FMM(P=4, ncrit=8)
    xs = [unit_cube(n, 10 + i) for i, n in enumerate(sizes)]
    print(f"[gpu] forest of {len(sizes)}", flush=True)
    for ys in (xs, xs[::-1]):
        got = f.evaluate_batch(ys)
        for y, g in zip(ys[:12], got):
            f.set_bodies(y)
            f.evaluate()
            # The same lists, summed in another order.
            assert rel_l2(np.asarray(g), f.results()) < 1e-12 or len(y) == 1
    f.close()
