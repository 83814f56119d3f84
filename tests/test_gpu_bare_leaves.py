"""Leaves that are in no P2P list, not even their own: where a leaf's centre lies
off its parent's by more than the parent's radius, the traversal takes the two
for well separated.  Bounds from the caller that do not enclose the bodies do
that, and centres rounded far from the origin.  The results of such a leaf's
bodies start from zero, whatever the handle held before, also for new charges
on the kept lists.

Bar: bit for bit between handles with another past (every pair on the per-pair
kernel, whose order does not change)."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import unit_cube

pytestmark = pytest.mark.gpu


def lattice(edge, far):
    g = np.stack(np.meshgrid(*[np.arange(edge)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return np.concatenate([g + far, np.random.default_rng(edge).uniform(-1, 1, (edge ** 3, 1))], axis=1)


CASES = {
    "bounds inside the bodies": (unit_cube(3000, 1), dict(P=6, ncrit=16), (np.full(3, -0.2), np.full(3, 0.3))),
    "the same, mixed": (unit_cube(3000, 1), dict(P=6, ncrit=16, precision="mixed"),
                        (np.full(3, -0.2), np.full(3, 0.3))),
    "rounded centres": (lattice(12, 2.0 ** 52), dict(P=4, theta=0.5, ncrit=1), None),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("updown", ["levels", "cells"])
def test_results_do_not_depend_on_the_past(name, updown, monkeypatch):
    x, kw, bounds = CASES[name]
    monkeypatch.setenv("EXAFMM_HIP_M2L", "pairs")
    monkeypatch.setenv("EXAFMM_HIP_UPDOWN", updown)
    res = []
    for seed in (1, 2):
        f = X.FMM(**kw)
        f.set_bodies(unit_cube(len(x), seed))
        f.evaluate()
        print(f"[gpu] {name}, {updown}, past {seed}", flush=True)
        f.set_bodies(x)
        b = f.get_bounds()
        f.build_tree(bounds or b)
        f.upward_pass()
        f.traverse()
        f.downward_pass()
        r = [f.results()]
        for scale in (2.0, 1.0, 1.0):
            f.evaluate_charges(scale * x[:, 3])
            r.append(f.results())
        res.append(r)
        f.close()
    if updown == "levels":
        assert (res[0][0] == 0).all(1).any()  # such leaves are there
    for a, b in zip(*res):
        assert np.array_equal(a, b)
    for r in res[0][2:]:
        assert np.array_equal(r, res[0][0])
