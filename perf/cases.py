"""Performance cases: what a user of the library has it do, over the range of
sizes, orders, trees, boundary conditions, bases and precisions it takes.

A case names one way of calling the library ("kind") and its settings:

  evaluate   new positions on the device, one FMM evaluation, results read on
             the device in tree order (a time step of a program that keeps
             its particles on the GPU)
  host       the same on host arrays, results back in the caller's order
  passes     host arrays through the pass-level calls, in the order of the
             reference's driver
  periodic   lattice in a periodic box: evaluation, dipole and its correction
  charges    new charges on kept positions (an iterative solver's step)
  batch      many independent systems on host arrays in one call
  ewald      tree build and Ewald summation on a lattice in a periodic box

Mixed-precision results are taken as float32, as a program that asks for that
form keeps its forces.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), os.pardir, "exafmm-dev_amd"))

import exafmm_hip  # noqa: E402

CYCLE = 2 * math.pi  # edge of the periodic box
FIRST = 2048         # leading results (tree order) that are checked by direct summation in large systems
WHOLE = 1 << 17      # systems up to this size are checked whole


def case(name, kind, n, P, data="cube", builder="uniform", precision="fp64", theta=0.4, ncrit=64, basis="spherical",
         images=0, systems=1):
    """`n`: bodies; lattice edge for lattices; bodies of the largest system for batches."""
    return dict(name=name, kind=kind, n=n, P=P, data=data, builder=builder, precision=precision, theta=theta,
                ncrit=ncrit, basis=basis, images=images, systems=systems)


def listed():
    return [
        # A small cluster evaluated from host arrays: launches and host waits are all of it.
        case("cube_2k_host", "host", 2000, 6),
        # A driver written like the reference's examples/serial.cxx, on a surface distribution and the adaptive tree.
        case("sphere_20k_passes", "passes", 20011, 8, data="sphere", builder="adaptive"),
        # A time step of a middle-sized particle code that keeps forces in single precision.
        case("cube_100k_mixed", "evaluate", 100003, 10, precision="mixed"),
        # The benchmark workload, in both forms.
        case("cube_1m", "evaluate", 1 << 20, 10),
        case("cube_1m_mixed", "evaluate", 1 << 20, 10, precision="mixed"),
        # Strongly clustered bodies: gravity at high order in the mixed form, and the largest system.
        case("plummer_250k_mixed", "evaluate", 250007, 12, data="plummer", builder="adaptive", precision="mixed"),
        case("plummer_4m", "evaluate", 1 << 22, 8, data="plummer", builder="adaptive"),
        # Ionic crystals under periodic boundary conditions, in both bases.
        case("periodic_64", "periodic", 64, 10, data="lattice", theta=0.35, images=3),
        case("periodic_48_cartesian", "periodic", 48, 6, data="lattice", theta=0.35, images=3, basis="cartesian"),
        # A boundary-integral solver's iteration: fixed points on a surface, a new charge vector.
        case("charges_500k", "charges", 500009, 8, data="sphere"),
        # Many small independent systems, half cubes, half spheres.
        case("batch_32", "batch", 16384, 8, data="mixed", theta=0.5, systems=32),
        # The Ewald sum that periodic results are checked with.
        case("ewald_32", "ewald", 32, 10, data="lattice", theta=0.35, images=3),
    ]


def log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["host", "passes", "evaluate", "evaluate", "evaluate", "periodic", "charges", "batch", "ewald"])
    P = rng.choice([4, 6, 8, 10, 12])
    precision = rng.choice(["fp64", "fp64", "mixed"])
    theta = rng.choice([0.35, 0.4, 0.5])
    data = rng.choice(["cube", "sphere", "plummer"])
    builder = "adaptive" if data == "plummer" else rng.choice(["uniform", "uniform", "adaptive"])
    ncrit = rng.choice([32, 64, 64, 128])
    if kind in ("host", "passes"):
        n = log_uniform(rng, 1000, 60000)
    elif kind == "evaluate":
        n = log_uniform(rng, 4000, 1 << 20 if P <= 10 and theta >= 0.4 else 1 << 18)
    elif kind == "charges":
        n = log_uniform(rng, 16000, 1 << 19)
    if kind in ("host", "passes", "evaluate", "charges"):
        return case("", kind, n, P, data, builder, precision, theta, ncrit)
    if kind == "batch":
        return case("", kind, log_uniform(rng, 4096, 32768), P, "mixed", "uniform", precision, theta, ncrit,
                    systems=rng.randint(8, 48))
    if kind == "periodic":
        basis = rng.choice(["spherical", "spherical", "cartesian"])
        if basis == "cartesian":
            return case("", kind, rng.randint(16, 48), rng.choice([4, 6]), "lattice", "uniform", "fp64", 0.4, 64,
                        basis, images=rng.randint(2, 4))
        return case("", kind, rng.randint(16, 64), P, "lattice", builder, precision, max(theta, 0.4), 64,
                    images=rng.randint(2, 4))
    return case("", "ewald", rng.randint(12, 32), 10, "lattice", "uniform", "fp64", 0.35, ncrit, images=3)


def num_bodies(c):
    return c["n"] ** 3 if c["data"] == "lattice" else c["n"]


def bodies(data, n, gen):
    """(n, 4) double x, y, z, q on the GPU."""
    dev = gen.device

    def uniform(*shape):
        return torch.rand(*shape, dtype=torch.float64, device=dev, generator=gen)

    def directions(m):
        v = torch.randn(m, 3, dtype=torch.float64, device=dev, generator=gen)
        return v / v.norm(dim=1, keepdim=True)

    if data == "lattice":  # rock salt with every ion moved by up to a quarter of the spacing; n = edge
        h = CYCLE / n
        g = torch.stack(torch.meshgrid(*[torch.arange(n, device=dev)] * 3, indexing="ij"), -1).reshape(-1, 3)
        x = (g + 0.5) * h + (uniform(n ** 3, 3) - 0.5) * (0.5 * h)
        return torch.cat([x, (1.0 - 2.0 * (g.sum(1) % 2))[:, None]], 1).contiguous()
    if data == "plummer":  # scale radius 1, cut at radius 10, equal masses
        top = (10.0 ** 2 / (1 + 10.0 ** 2)) ** 1.5  # mass fraction inside the cut
        r = 1.0 / torch.sqrt((uniform(n) * top).clamp_min(1e-12) ** (-2.0 / 3.0) - 1.0)
        return torch.cat([directions(n) * r[:, None], torch.full((n, 1), 1.0 / n, dtype=torch.float64, device=dev)],
                         1).contiguous()
    x = directions(n) if data == "sphere" else 2 * uniform(n, 3) - 1
    return torch.cat([x, charges(n, gen)[:, None]], 1).contiguous()


def charges(n, gen):
    q = torch.rand(n, dtype=torch.float64, device=gen.device, generator=gen) - 0.5
    return (q - q.mean()) / n


def inputs(c, seed):
    """The case's arrays on the GPU: bodies, and for `charges` the new charges; for `batch` the list of systems."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if c["kind"] == "batch":
        # Sizes spread evenly over the logarithm of a factor of 16.
        sizes = [int(c["n"] * 16.0 ** -((0.618034 * i) % 1.0)) for i in range(c["systems"])]
        return [bodies("cube" if i % 2 == 0 else "sphere", m, gen) for i, m in enumerate(sizes)]
    x = bodies(c["data"], c["n"], gen)
    return (x, charges(x.shape[0], gen)) if c["kind"] == "charges" else x


def prepare(c, seed):
    fmm = exafmm_hip.FMM(P=c["P"], theta=c["theta"], ncrit=c["ncrit"], images=c["images"], cycle=CYCLE,
                         builder=c["builder"], precision=c["precision"], basis=c["basis"])
    s = dict(kind=c["kind"], fmm=fmm, mixed=c["precision"] == "mixed", x=inputs(c, seed))
    if c["kind"] in ("host", "passes"):
        s["x"] = s["x"].cpu().numpy()
    elif c["kind"] == "batch":
        s["x"] = [v.cpu().numpy() for v in s["x"]]
    elif c["kind"] == "charges":
        s["x"], s["q"] = s["x"]
    torch.cuda.synchronize()
    if c["kind"] == "charges":  # the geometry that the solver iterates on
        fmm.set_bodies_device(s["x"].shape[0], s["x"].data_ptr())
        fmm.evaluate()
    return s


class DeviceArray:
    """An (n, 4) double array at a device address, for torch.as_tensor."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n, 4), typestr="<f8", data=(ptr, False), version=2)


def device_results(s):
    """Results in tree order, copied into the program's own array: the library's lives until its next evaluation or
    the end of the handle."""
    fmm = s["fmm"]
    p = exafmm_hip.ctypes.c_void_p()
    fmm._check(fmm.lib.exafmm_hip_results_device(fmm.h, exafmm_hip.ctypes.byref(p)), "results_device")
    r = torch.as_tensor(DeviceArray(p.value, fmm.n), device="cuda")
    r = r.to(torch.float32) if s["mixed"] else r.clone()
    return (r,) if fmm.n <= WHOLE else (r[:FIRST], r[FIRST:])


def host_results(s, r):
    return r.astype(np.float32) if s["mixed"] else r


def run(s):
    fmm, x = s["fmm"], s["x"]
    if s["kind"] in ("evaluate", "periodic", "charges"):
        # The library works on its own streams: the last step's results must have been read before it starts.
        torch.cuda.current_stream().synchronize()
    if s["kind"] == "evaluate":
        fmm.set_bodies_device(x.shape[0], x.data_ptr())
        fmm.evaluate()
        return device_results(s)
    if s["kind"] == "host":
        fmm.set_bodies(x)
        fmm.evaluate()
        return host_results(s, fmm.results())
    if s["kind"] == "passes":
        fmm.set_bodies(x)
        fmm.build_tree(fmm.get_bounds())
        fmm.upward_pass()
        fmm.traverse()
        fmm.downward_pass()
        return host_results(s, fmm.results())
    if s["kind"] == "periodic":
        fmm.set_bodies_device(x.shape[0], x.data_ptr())
        fmm.evaluate()
        fmm.dipole_correction(fmm.dipole(), x.shape[0], CYCLE)
        return device_results(s)
    if s["kind"] == "charges":
        fmm._check(fmm.lib.exafmm_hip_evaluate_charges_device(fmm.h, fmm.n, s["q"].data_ptr()), "evaluate_charges")
        return device_results(s)
    if s["kind"] == "batch":
        return host_results(s, np.concatenate(fmm.evaluate_batch(x)))
    fmm.set_bodies_device(x.shape[0], x.data_ptr())
    fmm.get_bounds()
    fmm.build_tree()
    return fmm.ewald(11, 10 / CYCLE, 0.25 / math.pi, CYCLE / 2, CYCLE)


def num_waves(ksize):
    k = range(-ksize, ksize + 1)
    return (sum(a * a + b * b + d * d <= ksize * ksize for a in k for b in k for d in k) - 1) // 2


def fmm_flops(n, P, theta, ncrit, basis):
    """Body pairs at 20 and cell pairs at the multiply-adds of the translation, 74 near leaves per leaf and 179
    separated cells per cell at theta = 0.4 (counted on the uniform cube), fewer in small systems."""
    depth = 1 + int(math.log(n // ncrit) / math.log(8)) if n >= ncrit else 0
    leaves = 8.0 ** depth
    cells = leaves * 8 / 7
    wider = (0.4 / theta) ** 3
    near = n * min(n, 74 * wider * n / leaves)
    far = cells * max(0.0, min(leaves - 74 * wider, 179 * wider))
    terms = {4: 140, 6: 924, 8: 3432}[P] if basis == "cartesian" else 8 * P * (P + 1) ** 2 * (P + 2) // 12
    return 20 * near + terms * far


def work(c):
    if c["kind"] == "batch":
        n = c["n"] * 15 / 16 / math.log(16)  # mean size
        return {"bytes": 64 * n * c["systems"],
                "flops": c["systems"] * fmm_flops(int(n), c["P"], c["theta"], c["ncrit"], c["basis"])}
    n = num_bodies(c)
    if c["kind"] == "ewald":  # pairs within half a box edge at 60, body-wave products at 8 there and 12 back
        return {"bytes": 64 * n, "flops": n * n * (math.pi / 6) * 60 + n * num_waves(11) * 20}
    out = 16 if c["precision"] == "mixed" else 32
    f = fmm_flops(n, c["P"], c["theta"], c["ncrit"], c["basis"])
    return {"bytes": ((8 if c["kind"] == "charges" else 32) + out) * n, "flops": f}


def direct(x, t):
    """Potential and gradient at t of the bodies x by plain summation."""
    out = torch.empty(t.shape[0], 4, dtype=torch.float64, device=x.device)
    rows = max(1, (1 << 26) // x.shape[0])
    for i in range(0, t.shape[0], rows):
        d = [t[i:i + rows, k, None] - x[None, :, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        inv = torch.where(r2 > 0, r2, math.inf).rsqrt()
        f = x[None, :, 3] * inv
        out[i:i + rows, 0] = f.sum(1)
        f *= inv * inv
        for k in range(3):
            out[i:i + rows, 1 + k] = -(d[k] * f).sum(1)
    return out


def tree_order(x, ncrit):
    """Order of the bodies in the uniform tree: Morton keys on the grid that the bounds and ncrit give."""
    n = x.shape[0]
    depth = 1 + int(math.log(n // ncrit) / math.log(2.0) / 3) if n >= ncrit else 0
    lo, hi = x[:, :3].amin(0), x[:, :3].amax(0)
    mid = (lo + hi) / 2
    size = np.float32(2 * (max((hi - mid).max().item(), (mid - lo).max().item()) * 1.00001) / 2 ** depth)
    cell = ((x[:, :3] - lo) / float(size)).long()
    key = torch.zeros(n, dtype=torch.int64, device=x.device)
    for b in range(depth):
        for k in range(3):
            key |= ((cell[:, k] >> b) & 1) << (3 * b + k)
    return torch.sort(key, stable=True).indices


def ewald_sum(x, ksize, alpha, sigma, cutoff):
    n = x.shape[0]
    k = torch.arange(-ksize, ksize + 1, dtype=torch.float64, device=x.device)
    w = torch.stack(torch.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)
    k2 = (w * w).sum(1)
    w, k2 = w[(k2 > 0) & (k2 <= ksize * ksize)], k2[(k2 > 0) & (k2 <= ksize * ksize)]
    s, q = 2 * math.pi / CYCLE, x[:, 3]
    out = torch.zeros(n, 4, dtype=torch.float64, device=x.device)
    coef = 0.25 / math.pi ** 2 / sigma / CYCLE * torch.exp(-k2 * (s * s / (4 * alpha * alpha))) / k2
    for i in range(0, w.shape[0], 512):  # both half spaces: half the half-space coefficient each
        v = w[i:i + 512]
        th = (x[:, :3] @ v.T) * s
        c, sn = torch.cos(th), torch.sin(th)
        a, b = coef[i:i + 512] * (q @ c), coef[i:i + 512] * (q @ sn)
        out[:, 0] += (c * a + sn * b).sum(1)
        out[:, 1:] -= ((sn * a - c * b) @ v) * s
    rows = max(1, (1 << 25) // n)
    for i in range(0, n, rows):
        d = [x[i:i + rows, j, None] - x[None, :, j] for j in range(3)]
        d = [v - CYCLE * torch.round(v / CYCLE) for v in d]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        on = (r2 > 0) & (r2 < cutoff * cutoff)
        r = torch.sqrt(torch.where(on, r2, 1.0))
        e = torch.erfc(alpha * r)
        f = torch.where(on, q[None, :], 0.0)
        out[i:i + rows, 0] += (f * e / r).sum(1)
        f = f * (2 / math.sqrt(math.pi) * alpha * torch.exp(-alpha * alpha * r * r) + e / r) / (r * r)
        for j in range(3):
            out[i:i + rows, 1 + j] -= (f * d[j]).sum(1)
    out[:, 0] -= 2 / math.sqrt(math.pi) * alpha * q
    return out


def exact(c, seed):
    """Direct sums (the Ewald sum for `ewald`); none where images of the box or the adaptive order would have to be
    followed."""
    v = inputs(c, seed)
    if c["kind"] == "batch":
        return torch.cat([direct(x, x) for x in v]).cpu().numpy()
    if c["kind"] in ("host", "passes"):
        return direct(v, v).cpu().numpy()
    if c["kind"] == "ewald":
        return ewald_sum(v, 11, 10 / CYCLE, 0.25 / math.pi, CYCLE / 2).cpu().numpy()
    if c["kind"] == "periodic" or c["builder"] == "adaptive":
        return None
    if c["kind"] == "charges":
        v = torch.cat([v[0][:, :3], v[1][:, None]], 1)
    t = v[tree_order(v, c["ncrit"])]
    if t.shape[0] <= WHOLE:
        return (direct(v, t),)
    return direct(v, t[:FIRST]), None
