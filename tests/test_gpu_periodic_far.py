"""Periodic far field by lattice sums, and the Cartesian kernels of each
order, against the oracle: every order of both bases, one to four image
levels, MASS mode, leaves of one body to more than a staged chunk (64), and
targets with fewer pairs than lanes and several rounds of them.

Bar: 1e-12 of the oracle, relative to the largest coefficient of L and in
the relative L2 norm of the results; M of the Cartesian basis bit for bit."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,P,images,mass,n,ncrit,builder", [
    ("spherical", 4, 2, False, 700, 30, "uniform"), ("spherical", 6, 4, False, 900, 64, "adaptive"),
    ("spherical", 8, 3, True, 900, 64, "uniform"), ("spherical", 10, 1, False, 700, 64, "uniform"),
    ("spherical", 12, 3, False, 1200, 64, "uniform"), ("cartesian", 4, 2, False, 700, 20, "uniform"),
    ("cartesian", 4, 0, True, 3000, 100, "adaptive"), ("cartesian", 6, 4, True, 900, 64, "uniform"),
    ("cartesian", 6, 0, False, 3000, 8, "adaptive"), ("cartesian", 6, 3, False, 1500, 200, "uniform"),
    ("cartesian", 8, 3, False, 900, 64, "uniform"), ("cartesian", 8, 1, True, 900, 40, "uniform")])
def test_far_field_orders(basis, P, images, mass, n, ncrit, builder):
    print(f"[gpu] {basis} P={P} images={images} mass={mass} n={n} ncrit={ncrit} {builder}", flush=True)
    rng = np.random.default_rng(n + P)
    q = rng.uniform(0.1, 1, n) if mass else rng.uniform(-1, 1, n)
    x = np.concatenate([rng.uniform(-np.pi, np.pi, (n, 3)), q[:, None] / n], axis=1)
    f = X.FMM(P=P, ncrit=ncrit, images=images, mass=mass, basis=basis, builder=builder)
    f.set_bodies(x)
    f.evaluate()
    o = run_oracle(x, P=P, ncrit=ncrit, images=images, mass=mass, basis=basis, adaptive=builder == "adaptive")
    c, oc = f.cells(), o.cells()
    if basis == "cartesian":
        assert np.array_equal(c["M"].real, oc["M"].real)
    assert np.abs(c["L"] - oc["L"]).max() <= 1e-12 * np.abs(oc["L"]).max()
    ob = o.bodies()
    ref = np.empty_like(ob["trg"])
    ref[ob["ibody"]] = ob["trg"]
    r = f.results()
    assert rel_l2(r[:, 0], ref[:, 0]) < 1e-12
    assert rel_l2(r[:, 1:], ref[:, 1:]) < 1e-12
    f.close()
