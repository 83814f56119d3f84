"""What a handle does after a call that was refused.

* A tree whose bounds have no extent is refused before anything is written: the
  tree there was goes on.  One that turns out too deep is refused after the old
  one is gone: the passes ask for a new one.
Bar: bit-identical to a handle that never met the refusal."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import unit_cube

pytestmark = pytest.mark.gpu


def passes(f):
    f.upward_pass()
    f.traverse()
    f.downward_pass()
    return f.results()


def fresh(x, **kw):
    f = X.FMM(**kw)
    f.set_bodies(x)
    f.build_tree(f.get_bounds())
    r = passes(f)
    f.close()
    return r


def test_refused_tree():
    x, kw = unit_cube(3000, 1), dict(P=4, ncrit=20, builder="adaptive")
    want = fresh(x, **kw)
    f = X.FMM(**kw)
    f.set_bodies(x)
    f.build_tree(f.get_bounds())
    print("[gpu] bounds without extent", flush=True)
    with pytest.raises(X.ExafmmError, match="degenerate bounds"):
        f.build_tree((np.zeros(3), np.zeros(3)))
    assert np.array_equal(passes(f), want)
    print("[gpu] a tree too deep", flush=True)
    with pytest.raises(X.ExafmmError, match="deeper than 20 levels"):
        f.build_tree((np.full(3, -1e9), np.full(3, 1e9)))
    for call in (f.upward_pass, f.traverse, f.results, f.cells):
        with pytest.raises(X.ExafmmError):
            call()
    f.build_tree(f.get_bounds())
    assert np.array_equal(passes(f), want)
    f.close()


@pytest.mark.parametrize("kw", [dict(P=8, ncrit=64), dict(P=6, ncrit=64, builder="adaptive", precision="mixed"),
                                dict(P=4, ncrit=64, basis="cartesian")])
@pytest.mark.parametrize("then", ["passes", "evaluate", "passes of the same tree"])
def test_refused_evaluation(kw, then, monkeypatch):
    x, big = unit_cube(20000, 2), unit_cube(60000, 3)
    f = X.FMM(**kw)
    f.set_bodies(x)
    limit = f.build_tree(f.get_bounds()) + 1
    f.close()
    want = fresh(x, **kw)
    monkeypatch.setenv("EXAFMM_HIP_MAX_CELLS", str(limit))
    f = X.FMM(**kw)
    f.set_bodies(big)
    print(f"[gpu] evaluation of more than {limit} cells refused, then {then}", flush=True)
    with pytest.raises(X.ExafmmError, match="cells"):
        f.evaluate()
    if then == "passes of the same tree":
        f.upward_pass()
        with pytest.raises(X.ExafmmError, match="cells"):
            f.traverse()
    f.set_bodies(x)
    if then == "evaluate":
        f.evaluate()
        got = f.results()
    else:
        f.build_tree(f.get_bounds())
        got = passes(f)
    assert np.array_equal(got, want)
    f.close()
