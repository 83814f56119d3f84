"""What get_stats says of the M2L: nothing of an earlier system, and as many
offsets as the list has."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import unit_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_no_pairs_after_a_larger_system(precision):
    f = X.FMM(P=6, ncrit=64, precision=precision)
    print("[gpu] statistics of one leaf after 20000 bodies", flush=True)
    f.set_bodies(unit_cube(20000, 1))
    f.evaluate()
    s = f.stats()
    names = ("num_m2l_lattice", "num_m2l_offsets", "num_m2l_tiles", "num_m2l_steps", "t_m2l_mfma")
    assert all(s[k] > 0 for k in names)
    f.set_bodies(unit_cube(30, 2))
    f.evaluate()
    s = f.stats()
    assert s["num_m2l_pairs"] == 0
    assert {k: s[k] for k in names + ("t_m2l_pairs",)} == dict.fromkeys(names + ("t_m2l_pairs",), 0)
    f.close()


def test_offsets_of_the_list():
    f = X.FMM(P=4, ncrit=32)
    for n in (20000, 1500, 9000):  # one handle: it knows the offsets of the larger trees
        f.set_bodies(unit_cube(n, n))
        f.evaluate()
        c, l, s = f.cells(), f.lists(), f.stats()
        print(f"[gpu] {n} bodies, {s['num_m2l_offsets']} offsets", flush=True)
        assert s["num_m2l_lattice"] == s["num_m2l_pairs"] == len(l["m2l_i"])
        # In quarters of the target's width, which is twice its distance to the parent's centre in any
        # coordinate (the residues modulo 4 tell the source's level).
        up = np.abs(c["X"] - c["X"][c["iparent"]]).max(1)
        i, j = l["m2l_i"], l["m2l_j"]
        d = np.rint((c["X"][i] - c["X"][j]) / (0.5 * up[i])[:, None]).astype(int)
        assert s["num_m2l_offsets"] == len(np.unique(d, axis=0))
    f.close()
