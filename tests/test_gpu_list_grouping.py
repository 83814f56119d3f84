"""Grouping of the interaction lists by target: the P2P list that the library
returns is the oracle's pair set, grouped, at the lengths where the grouping
changes method: targets with at most 64 entries, up to 1024, and beyond (a
few large leaves next to thousands of small ones), and target counts over a
scan chunk (4096).  The order within a target is the emission order, which is
fixed: two handles, and a handle's first (host-driven) and second
(device-driven) traversal, return the same arrays."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import plummer, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


def clustered(n, m):
    """n bodies in a tiny clump inside the box of a few distant ones."""
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.uniform(-1, 1, (m, 3)), 0.3 + 0.02 * rng.uniform(-1, 1, (n, 3))])
    return np.concatenate([x, rng.uniform(-1, 1, (n + m, 1))], axis=1)


@pytest.mark.parametrize("name,x,kw", [
    ("one leaf", unit_cube(10, 1), dict(ncrit=64)),
    ("two levels", unit_cube(500, 2), dict(ncrit=64)),
    ("one body per leaf", unit_cube(3000, 3), dict(ncrit=1, builder="adaptive", theta=0.6)),
    ("wide lists", unit_cube(4000, 4), dict(ncrit=2, theta=0.15)),
    ("longest lists", clustered(6000, 40), dict(ncrit=2, theta=0.1, builder="adaptive")),
    ("many targets", unit_cube(40000, 5), dict(ncrit=8)),
    ("adaptive", plummer(20000, 6), dict(ncrit=30, builder="adaptive")),
    ("mutual", unit_cube(6000, 7), dict(ncrit=16, mutual=1))])
def test_grouped_lists(name, x, kw):
    f = X.FMM(P=4, **kw)
    f.set_bodies(x)
    f.evaluate()
    first = f.lists()
    per = np.bincount(first["p2p_i"])
    print(f"[gpu] {name}: {len(first['p2p_i'])} entries, up to {per.max()} per target", flush=True)
    if name == "longest lists":
        assert per.max() > 1024
    assert np.all(np.diff(first["p2p_i"]) >= 0)
    kw = dict(kw)
    adaptive = kw.pop("builder", "uniform") == "adaptive"
    o = run_oracle(x, P=4, adaptive=adaptive, **kw).lists()
    key = lambda i, j: np.sort(i.astype(np.int64) << 32 | j)  # noqa: E731
    for a, b in (("p2p_i", "p2p_j"), ("m2l_i", "m2l_j")):
        assert np.array_equal(key(first[a], first[b]), key(o[a], o[b]))
    f.evaluate()
    second = f.lists()
    f.close()
    for k in first:
        assert np.array_equal(first[k], second[k]), k
