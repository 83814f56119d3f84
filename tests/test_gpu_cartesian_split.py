"""The Cartesian multipoles beside the traversal (inside one evaluation) against
the passes one after another: the same arithmetic in the same order, so cells,
radii, multipoles, expansions and results agree to the bit."""
import numpy as np
import pytest

import exafmm_hip as X

pytestmark = pytest.mark.gpu


# One leaf and no pair; fewer bodies than a leaf holds; a level of one parent;
# a deep ragged tree; images; radii without the rmax bound.
@pytest.mark.parametrize("n,P,builder,kw", [
    (1, 4, "uniform", {}), (40, 6, "adaptive", {}), (300, 8, "uniform", {}),
    (5001, 4, "adaptive", {}), (9000, 6, "uniform", dict(images=2, cycle=2.0)),
    (9000, 6, "adaptive", dict(useRmax=0)), (3000, 8, "adaptive", dict(mass=1)),
])
def test_evaluate_equals_passes(n, P, builder, kw):
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.uniform(-1, 1, (n, 3)) ** 3, rng.uniform(0.1, 1, (n, 1))], 1)
    out = []
    for whole in (True, False):
        f = X.FMM(P=P, theta=0.45, ncrit=48, builder=builder, basis="cartesian", **kw)
        for _ in range(2):  # the second on kept buffers
            f.set_bodies(x)
            if whole:
                f.evaluate()
            else:
                f.get_bounds()
                f.build_tree()
                f.upward_pass()
                f.traverse()
                f.downward_pass()
        c = f.cells()
        out.append([c[k] for k in ("icell", "nbody", "R", "X", "M", "L")] + [f.results()])
        f.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
