"""Trees so far from the origin that cell centres are rounded to whole numbers a
cell apart: integer positions from 2^52 on, one body to a leaf, where sibling
leaves have one centre.  Every M2L pair counts: the lattice M2L against every
pair on the per-pair kernel (the same lists).  The larger tree has more cells on
a level than one workgroup orders.

Bar: 1e-12, the sums of the same terms in another order."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge,builder", [(12, "adaptive"), (12, "uniform"), (44, "adaptive")])
@pytest.mark.parametrize("far", [2.0 ** 52, 2.0 ** 45])
def test_rounded_centres(edge, builder, far, monkeypatch):
    g = np.stack(np.meshgrid(*[np.arange(edge)] * 3, indexing="ij"), -1).reshape(-1, 3)
    q = np.random.default_rng(edge).uniform(-1, 1, (edge ** 3, 1))
    x = np.concatenate([g + far, q], axis=1)
    res = []
    for m2l in ("lattice", "pairs"):
        monkeypatch.setenv("EXAFMM_HIP_M2L", m2l)
        f = X.FMM(P=4, theta=0.5, ncrit=1, builder=builder)
        f.set_bodies(x)
        f.evaluate()
        s = f.stats()
        print(f"[gpu] {builder}, {edge}^3 from {far:g}, {m2l}: {s['num_m2l_lattice']} of {s['num_m2l_pairs']} pairs "
              "on the lattice", flush=True)
        assert s["num_m2l_pairs"] > 0
        res.append(f.results())
        f.close()
    assert rel_l2(res[0], res[1]) < 1e-12


@pytest.mark.parametrize("lo,hi", [(-0.2, 0.3), (-1.5, 1.2)])
def test_bounds_asked_for_after_the_build(lo, hi):
    """The tree keeps the bounds it was built from, whatever get_bounds computes before its lists are made."""
    x = np.random.default_rng(5).uniform(-1, 1, (3000, 4))
    res = []
    for ask in (False, True):
        f = X.FMM(P=6, ncrit=16)
        f.set_bodies(x)
        f.build_tree((np.full(3, lo), np.full(3, hi)))
        f.upward_pass()
        print(f"[gpu] bounds {lo} to {hi} from the caller, asked for again: {ask}", flush=True)
        if ask:
            f.get_bounds()
        f.traverse()
        f.downward_pass()
        res.append(f.results())
        f.close()
    assert rel_l2(res[1], res[0]) < 1e-12
