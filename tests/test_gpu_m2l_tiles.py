"""Lattice M2L with so many target tiles that their number is counted on the
device instead of bounded by the parents': trees of one body to a leaf, whose
parents have a third of the children that they could have, then a small tree on
the same handle.  Against every pair on the per-pair kernel (the same lists).

Bar: 1e-12, the sums of the same terms in another order."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2, unit_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("builder", ["uniform", "adaptive"])
def test_counted_tiles(builder, monkeypatch):
    xs = [unit_cube(300000, 1), unit_cube(9000, 2), unit_cube(300000, 3)]
    res = {}
    for m2l in ("lattice", "pairs"):
        monkeypatch.setenv("EXAFMM_HIP_M2L", m2l)
        f = X.FMM(P=4, theta=0.7, ncrit=1, builder=builder)
        res[m2l] = []
        for x in xs:
            f.set_bodies(x)
            f.evaluate()
            s = f.stats()
            print(f"[gpu] {builder}, {m2l}: {s['num_cells']} cells, {s['num_m2l_tiles']} tiles, "
                  f"{s['num_m2l_lattice']} of {s['num_m2l_pairs']} pairs on the lattice", flush=True)
            res[m2l].append((s, f.results()))
        f.close()
    for (s, a), (_, b) in zip(res["lattice"], res["pairs"]):
        assert s["num_m2l_lattice"] > 0.9 * s["num_m2l_pairs"]
        # Tiles are full but for the last of each level and octant.
        assert s["num_m2l_tiles"] <= s["num_cells"] / 64 + 8 * s["num_levels"]
        assert rel_l2(a, b) < 1e-12
