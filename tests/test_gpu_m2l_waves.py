"""The per-pair M2L where every target has a wave of its own: more than 2048
targets with 16 pairs and more each and a million pairs in all (fewer and several
waves share a target).  Against the oracle.

Bar: FP64 1e-12 of the oracle's largest local coefficient; mixed 1e-6 of the
FP64 form (FP32 tables and products: 2^-24 per product, a few hundred per
coefficient of random sign)."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2, run_oracle, unit_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,n,ncrit,theta", [(4, 40000, 8, 0.4), (6, 36000, 8, 0.35)])
def test_one_wave_per_target(P, n, ncrit, theta, monkeypatch):
    monkeypatch.setenv("EXAFMM_HIP_M2L", "pairs")
    x = unit_cube(n, n + P)
    res = {}
    for precision in ("fp64", "mixed"):
        f = X.FMM(P=P, ncrit=ncrit, theta=theta, precision=precision)
        f.set_bodies(x)
        f.evaluate()
        s = f.stats()
        targets = len(np.unique(f.lists()["m2l_i"]))
        print(f"[gpu] P={P} n={n} {precision}: {targets} targets, {s['num_m2l_pairs']} pairs", flush=True)
        assert s["num_m2l_lattice"] == 0
        assert targets > 2048 and s["num_m2l_pairs"] >= max(1 << 20, 16 * targets)
        res[precision] = (f.cells()["L"], f.results())
        f.close()
    o = run_oracle(x, P=P, ncrit=ncrit, theta=theta)
    oL = o.cells()["L"]
    assert np.abs(res["fp64"][0] - oL).max() <= 1e-12 * np.abs(oL).max()
    assert rel_l2(res["mixed"][1], res["fp64"][1]) < 1e-6
