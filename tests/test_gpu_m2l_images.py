"""M2L of pairs across one face of a periodic box on the matrix cores against
the per-pair kernel: trees of 3 to 5 levels (which levels take part), both
builders, box lengths near to and far from the bodies' extent, every form of
the coefficients, and one handle whose box, tree and levels change."""
import numpy as np
import pytest

import exafmm_hip as X
from helpers import rel_l2

pytestmark = pytest.mark.gpu


def box(n, seed, cycle=2 * np.pi):
    rng = np.random.default_rng(seed)
    q = rng.uniform(-0.5, 0.5, n)
    x = rng.uniform(-cycle / 2, cycle / 2, (n, 3))
    return np.concatenate([x, ((q - q.mean()) / n)[:, None]], axis=1)


def run(f, x):
    f.set_bodies(x)
    f.evaluate()
    return f.cells()["L"], f.results(), f.stats()


@pytest.mark.parametrize("P,n,ncrit,theta,cycle,builder,precision", [
    (4, 3000, 40, 0.5, 2 * np.pi, "uniform", "fp64"), (10, 20000, 32, 0.4, 2 * np.pi, "uniform", "fp64"),
    (12, 9000, 100, 0.5, 7.5, "uniform", "fp64"), (6, 40000, 8, 0.6, 6.9, "uniform", "fp64"),
    (8, 12000, 20, 0.4, 2 * np.pi, "adaptive", "fp64"), (8, 20000, 32, 0.4, 6.5, "uniform", "mixed"),
    (10, 500, 60, 0.4, 2 * np.pi, "uniform", "fp64")])
def test_image_pairs_match_per_pair(P, n, ncrit, theta, cycle, builder, precision, monkeypatch):
    print(f"[gpu] image M2L P={P} n={n} {builder} {precision}", flush=True)
    x = box(n, n)
    out = {}
    for mode in ("pairs", "lattice"):
        monkeypatch.setenv("EXAFMM_HIP_M2L", mode)
        f = X.FMM(P=P, theta=theta, ncrit=ncrit, images=2, cycle=cycle, builder=builder, precision=precision)
        out[mode] = run(f, x)
        f.close()
    (La, ra, sa), (Lb, rb, sb) = out["pairs"], out["lattice"]
    assert sa["num_m2l_pairs"] == sb["num_m2l_pairs"]
    print(f"[gpu]   {sb['num_m2l_lattice']} of {sb['num_m2l_pairs']} pairs, {sb['num_m2l_offsets']} offsets", flush=True)
    # Sums of the same terms in another order, in FP64 or with FP32 tables and
    # sums over one expansion (up to 110 terms of 6e-8 each).
    tol = 1e-12 if precision == "fp64" else 1e-5
    assert np.abs(Lb - La).max() <= tol * np.abs(La).max()
    assert rel_l2(rb, ra) < tol


def test_box_and_tree_change_on_one_handle():
    kw = dict(P=6, theta=0.5, ncrit=16, images=2)
    f = X.FMM(cycle=2 * np.pi, **kw)
    last = None
    for n, cycle in ((20000, 2 * np.pi), (20000, 7.0), (1500, 7.0), (90000, 6.5), (20000, 2 * np.pi)):
        f.set_config(cycle=cycle)
        x = box(n, n)
        got = run(f, x)[1]
        g = X.FMM(cycle=cycle, **kw)
        assert np.array_equal(got, run(g, x)[1])
        g.close()
        assert last is None or got.shape != last.shape or not np.array_equal(got, last)
        last = got
    f.close()
