"""Per-pair M2L with one and with several waves per target: every pair on the
per-pair kernel (EXAFMM_HIP_M2L=pairs) against the oracle, with few targets
(several waves share one; lists shorter than the waves too) and with more
targets than that rule takes (one wave each).

Bar: FP64 1e-12 of the oracle's largest local coefficient; mixed 1e-6 of the
FP64 form (FP32 tables and products: 2^-24 per product, a few hundred per
coefficient of random sign)."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,n,ncrit", [(4, 300, 8), (6, 2000, 64), (8, 700, 30), (10, 2500, 64), (12, 1500, 64),
                                       (8, 30000, 64), (12, 30000, 64)])
def test_pairs_against_oracle(P, n, ncrit, monkeypatch):
    monkeypatch.setenv("EXAFMM_HIP_M2L", "pairs")
    x = unit_cube(n, n + P)
    res = {}
    for precision in ("fp64", "mixed"):
        f = X.FMM(P=P, ncrit=ncrit, precision=precision)
        f.set_bodies(x)
        f.evaluate()
        s = f.stats()
        print(f"[gpu] P={P} n={n} {precision}: {s['num_cells']} cells, {s['num_m2l_pairs']} pairs", flush=True)
        assert s["num_m2l_lattice"] == 0
        res[precision] = (f.cells()["L"], f.results())
        f.close()
    o = run_oracle(x, P=P, ncrit=ncrit)
    oL = o.cells()["L"]
    assert np.abs(res["fp64"][0] - oL).max() <= 1e-12 * np.abs(oL).max()
    assert rel_l2(res["mixed"][1], res["fp64"][1]) < 1e-6
