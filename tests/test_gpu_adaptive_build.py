"""The adaptive tree against the oracle's, bit for bit, where the build changes
method: trees within the levels that one workgroup builds and beyond, a root
that is a leaf, leaves of up to 64, 1024 and more bodies (the sort of a leaf's
indices), coincident bodies, bodies on the cell faces, a handle whose last
tree was shallower (its shorter keys do not reach) or deeper, and trees that
the builder refuses."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import plummer, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


def check(f, x, ncrit, theta=0.4):
    f.set_bodies(x)
    f.evaluate()
    o = run_oracle(x, P=4, ncrit=ncrit, theta=theta, adaptive=True)
    c, oc = f.cells(), o.cells()
    for k in ("iparent", "ichild", "nchild", "ibody", "nbody", "icell", "X", "R"):
        assert np.array_equal(c[k], oc[k]), k
    b, ob = f.bodies(), o.bodies()
    assert np.array_equal(b["ibody"], ob["ibody"])
    assert np.array_equal(b["xyzq"], ob["xyzq"])
    return f.stats()["num_levels"]


def with_coincident(n, m):
    x = unit_cube(n, n)
    x[:m, :3] = x[0, :3]
    return x[np.random.default_rng(1).permutation(n)]


def on_faces(n):
    rng = np.random.default_rng(n)
    x = rng.integers(-8, 9, (n, 3)) / 8.0
    return np.concatenate([x, rng.uniform(-1, 1, (n, 1))], axis=1)


@pytest.mark.parametrize("name,x,ncrit", [
    ("root leaf", unit_cube(50, 1), 64), ("large root leaf", unit_cube(3000, 1), 4000),
    ("two levels", unit_cube(130, 2), 64), ("small", plummer(3000, 3), 30), ("large leaves", plummer(20000, 4), 900),
    ("larger leaves", unit_cube(20000, 5), 5000), ("onesweep keys", plummer(90000, 6), 64),
    ("one body per leaf", plummer(4000, 7), 1), ("coincident", with_coincident(3000, 40), 50),
    ("faces", on_faces(4000), 40)])
def test_tree_matches_oracle(name, x, ncrit):
    print(f"[gpu] adaptive build: {name}", flush=True)
    f = X.FMM(P=4, ncrit=ncrit, builder="adaptive")
    check(f, x, ncrit)
    check(f, x, ncrit)  # from the sizes of the last tree
    f.close()


def test_deeper_and_shallower_trees_on_one_handle():
    f = X.FMM(P=4, ncrit=20, builder="adaptive")
    deep = plummer(30000, 9)
    deep[:200, :3] *= 1e-3
    levels = [check(f, x, 20) for x in (unit_cube(2000, 8), deep, unit_cube(500, 8), deep, unit_cube(60000, 8))]
    print(f"[gpu] levels {levels}", flush=True)
    assert levels[1] > levels[0] + 2
    f.close()


def test_refused_trees():
    f = X.FMM(P=4, ncrit=20, builder="adaptive")
    x = unit_cube(400, 1)
    check(f, x, 20)
    f.set_bodies(with_coincident(400, 30))
    with pytest.raises(X.ExafmmError, match="deeper than 20 levels"):
        f.evaluate()
    y = x.copy()
    y[:, :3] = 0.5
    f.set_bodies(y)
    with pytest.raises(X.ExafmmError, match="degenerate bounds"):
        f.evaluate()
    check(f, x, 20)
    f.close()
