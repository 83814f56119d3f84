"""The mixed P2P's grid of half as many waves as leaves (trees of one to two
rounds of the resident grid with a longer M2L beside it) against one wave per
leaf: every target's sums run in the same order on any grid, so the results
agree to the bit, evaluated whole, pass by pass and for new charges."""
import numpy as np
import pytest

import exafmm_hip as X

pytestmark = pytest.mark.gpu


# Leaves: 4096, 3691 and 6077 (an odd number, and just inside the range on 256 CUs),
# 512 and 23116 (outside), and 4096 with a longer P2P (outside).
@pytest.mark.parametrize("n,P,ncrit,builder", [
    (33000, 8, 64, "uniform"), (9500, 6, 8, "adaptive"), (22400, 6, 8, "adaptive"),
    (5000, 8, 64, "uniform"), (40000, 6, 8, "uniform"), (90000, 4, 64, "uniform"),
])
def test_grid_does_not_matter(n, P, ncrit, builder, monkeypatch):
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.uniform(-1, 1, (n, 3)), rng.uniform(-0.5, 0.5, (n, 1))], 1)
    q = rng.uniform(-0.5, 0.5, n)
    out = []
    for one_wave in (False, True):
        if one_wave:
            monkeypatch.setenv("EXAFMM_HIP_P2P_WAVES", "0")
        f = X.FMM(P=P, theta=0.45, ncrit=ncrit, builder=builder, precision="mixed")
        f.set_bodies(x)
        f.evaluate()
        f.evaluate()  # the device-driven traversal
        r = [f.results().copy()]
        f.upward_pass()
        f.traverse()
        f.downward_pass()
        r.append(f.results().copy())
        f.evaluate_charges(q)
        f.evaluate_charges(q)  # the recorded graph
        r.append(f.results().copy())
        print(f"[gpu] n={n} P={P} leaves={len(np.unique(f.lists()['p2p_i']))}", flush=True)
        f.close()
        out.append(r)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
