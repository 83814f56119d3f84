"""FP64 P2P with several waves per leaf against the oracle, where a wave's share
of the list's bodies starts or ends in an unusual place: fewer bodies than
waves, shares inside one leaf, lists of more than 64 leaves (the search for the
start goes through several blocks of entries), one leaf that holds almost all
bodies, and periodic images (the own leaf in the list again, shifted)."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


def lump(n, m):
    x = unit_cube(n, n)
    x[:m, :3] = 0.9 + 0.01 * x[:m, :3]
    return x


@pytest.mark.parametrize("name,x,kw", [
    ("two bodies", unit_cube(2, 1), dict(ncrit=64)), ("fewer bodies than waves", unit_cube(5, 2), dict(ncrit=1)),
    ("one leaf", unit_cube(700, 3), dict(ncrit=1000)), ("long lists", unit_cube(2500, 4), dict(ncrit=4, theta=0.25)),
    ("long lists, four waves", unit_cube(20000, 5), dict(ncrit=24, theta=0.3)),
    ("lump", lump(1500, 1400), dict(ncrit=64)), ("lump, adaptive", lump(3000, 2500), dict(ncrit=300, adaptive=True)),
    ("images", unit_cube(600, 6), dict(ncrit=40, images=2, cycle=2.0))])
def test_teams_match_oracle(name, x, kw):
    print(f"[gpu] P2P teams: {name}", flush=True)
    kw = dict(theta=0.4) | kw
    adaptive = kw.pop("adaptive", False)
    f = X.FMM(P=6, builder="adaptive" if adaptive else "uniform", **kw)
    f.set_bodies(x)
    f.evaluate()
    o = run_oracle(x, P=6, adaptive=adaptive, **kw)
    b = o.bodies()
    ref = np.empty_like(b["trg"])
    ref[b["ibody"]] = b["trg"]
    # Same lists and terms, summed in another order.
    assert rel_l2(f.results(), ref) < 1e-12
    f.close()
