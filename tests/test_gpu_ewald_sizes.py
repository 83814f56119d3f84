"""Ewald summation against the oracle where its kernels change shape: wave
counts at the edges of the tiles of n (6) and of the staged bodies (64 up to
ksize 27, 16 above), leaves of 1 to 100 bodies (lane groups of 8 to 64, second
passes), source cells split over workgroups (few leaves) or not, the ancestor
walk (short cut-off) and a splitting parameter that underflows erfc.

Bar: 1e-12 (relative L2).  The oracle's own phases k.x carry an error of half
an ulp of |k.x| <= 2 pi sqrt(3) 28 (3e-14) per wave, and both sides sum up to
2000 pairs or 90000 waves in different orders (n eps at worst per sum of
one sign, 2e-13)."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2, run_oracle

pytestmark = pytest.mark.gpu
CYC = 2 * np.pi


@pytest.mark.parametrize("n,ncrit,ksize,alpha,cutoff", [
    (1, 64, 3, 10, 0.5), (65, 64, 1, 10, 0.5), (300, 8, 5, 10, 0.5), (300, 8, 6, 10, 0.14), (701, 64, 12, 10, 0.5),
    (777, 100, 27, 4, 0.3), (500, 200, 28, 10, 0.5), (2000, 16, 11, 10, 0.5), (1500, 30, 0, 60, 0.5)])
def test_ewald_shapes(n, ncrit, ksize, alpha, cutoff):
    print(f"[gpu] ewald n={n} ncrit={ncrit} ksize={ksize}", flush=True)
    rng = np.random.default_rng(n + ksize)
    x = np.concatenate([rng.uniform(0, CYC, (n, 3)), rng.uniform(-1, 1, (n, 1))], axis=1)
    args = (ksize, alpha / CYC, 0.25 / np.pi, cutoff * CYC, CYC)
    f = X.FMM(P=4, ncrit=ncrit, images=1, cycle=CYC)
    f.set_bodies(x)
    f.get_bounds()
    f.build_tree()
    e = f.ewald(*args)
    o = run_oracle(x, P=4, ncrit=ncrit, images=1, cycle=CYC)
    ref = o.ewald(*args)
    assert rel_l2(e[:, 0], ref[:, 0]) < 1e-12
    if n > 1:
        assert rel_l2(e[:, 1:], ref[:, 1:]) < 1e-12
    start = rng.uniform(-1, 1, (n, 4))  # added to what the caller's array holds
    got = f.ewald(*args, trg=start.copy())
    assert np.abs(got - start - e).max() <= 1e-14 * (1 + np.abs(e).max())
    f.close()
