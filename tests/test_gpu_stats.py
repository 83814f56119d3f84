"""What get_stats says of the M2L: nothing of an earlier system."""
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
