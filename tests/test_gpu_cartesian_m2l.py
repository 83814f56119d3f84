"""Cartesian M2L with a pair per lane, P = 8 in two kernels of outputs, against
the oracle's local expansions: lists of one pair up to several rounds of 64,
image pairs and the mass weighting.

A local coefficient is a sum of at most 120 terms per pair, rounded at 1.1e-16
each, over at most some thousand pairs: 1e-12 of the largest coefficient of its
degree holds with a margin of ten (derivatives of degree k grow as k!, so each
degree has its own bar)."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [4, 6, 8])
@pytest.mark.parametrize("n,ncrit,kw", [
    (60, 8, {}), (1500, 16, {}), (1500, 16, dict(images=2, cycle=2.0)), (700, 16, dict(mass=1)),
])
def test_local_expansions(P, n, ncrit, kw):
    rng = np.random.default_rng(n + P)
    x = np.concatenate([rng.uniform(-1, 1, (n, 3)) ** 3, rng.uniform(0.1, 1, (n, 1))], 1)
    f = X.FMM(P=P, theta=0.5, ncrit=ncrit, builder="adaptive", basis="cartesian", **kw)
    f.set_bodies(x)
    f.evaluate()
    o = run_oracle(x, P=P, theta=0.5, ncrit=ncrit, adaptive=True, basis="cartesian", **kw)
    got, want = f.cells()["L"].real, o.cells()["L"].real
    assert len(f.lists()["m2l_i"]) > 0
    for k in range(P):
        lo, hi = k * (k + 1) * (k + 2) // 6, (k + 1) * (k + 2) * (k + 3) // 6
        assert np.abs(got[:, lo:hi] - want[:, lo:hi]).max() <= 1e-12 * np.abs(want[:, lo:hi]).max(), k
    f.close()
