"""Wave part of the Ewald summation with few waves: fewer rows than partial
results the back transform splits into otherwise (ksize 1 to 3), and workgroups
of 64 and of 256 bodies.  Against the sum over the waves of one half space.

Bar: 1e-13 of the largest term's sum (n eps for n = 20000 terms of either sign
is 4e-12 at worst, sqrt(n) eps 3e-14 as a rule; the phases' error is an ulp of
2 pi)."""
import numpy as np
import pytest

import exafmm_hip as X

pytestmark = pytest.mark.gpu
CYC = 2 * np.pi


@pytest.mark.parametrize("ksize", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [1, 64, 65, 700, 16127, 16129, 20000])
def test_wave_part(n, ksize):
    print(f"[gpu] ewald waves, n={n} ksize={ksize}", flush=True)
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.uniform(0, CYC, (n, 3)), rng.uniform(-1, 1, (n, 1))], axis=1)
    alpha, sigma = 1.5, 0.25 / np.pi
    f = X.FMM(P=4, ncrit=64)
    f.set_bodies(x)
    f.get_bounds()
    f.build_tree()
    got = f.ewald(ksize, alpha, sigma, 1.0, CYC, 1)
    f.close()
    g = np.arange(-ksize, ksize + 1)
    k = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    k2 = (k ** 2).sum(1)
    k = k[(k2 <= ksize ** 2) & ((k[:, 0] > 0) | (k[:, 0] == 0) & (k[:, 1] > 0) | (k[:, 0] == 0) & (k[:, 1] == 0) &
                                (k[:, 2] > 0))]
    k2 = (k ** 2).sum(1)
    s = 2 * np.pi / CYC
    coef = 0.5 / np.pi ** 2 / sigma / CYC * np.exp(-k2 * s * s / (4 * alpha * alpha)) / k2
    ph = s * (x[:, :3] @ k.T)
    w = coef * (x[:, 3] @ np.exp(1j * ph))
    z = w * np.exp(-1j * ph)
    want = np.concatenate([z.real.sum(1)[:, None], s * (z.imag @ k)], axis=1)
    bound = np.abs(coef).sum() * np.abs(x[:, 3]).sum() * ksize
    assert np.abs(got - want).max() <= 1e-13 * bound
