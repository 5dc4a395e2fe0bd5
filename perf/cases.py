"""Performance cases of the treecode: what programs have it do, over the range
of sizes, distributions and options they use, each through the public entry
points (the Treecode class and the C ABI under it).

Kinds of case:

force   a host program asks for the forces on its particles: the particles go
        in from host arrays, the accelerations and potentials come back to the
        host in the program's own order (an integrator outside this library)
device  the same evaluation for a program whose particles are already on the
        GPU and which reads the results there
build   the tree without the walk: octree, moments and groups of particles on
        the GPU, copied there into arrays of the program's own (a program with
        its own walk or neighbour search)
step    a simulation: a few kick-drift-kick steps, then a snapshot
graph   the same with the captured step
train   minibatch training of the opening-angle network

`listed()` are the cases measured by name, `draw(rng)` gives further ones of
the same ranges, `prepare` makes what a program holds before the call, `run`
is one pass, `work` its unavoidable bytes and flops, and `exact` its result in
64 bits by direct summation where that is affordable.
"""
import ctypes
import math

import numpy as np
import torch

import bonsai2_amd as bt

# BT_BUF_* of include/bonsai2_amd.h
BUF_POS, BUF_ACC, BUF_CELLS, BUF_LEVELS = 0, 3, 6, 5
BUF_SIZE, BUF_MONO, BUF_QUAD0, BUF_QUAD1 = 7, 8, 9, 10
BUF_GROUPS, BUF_PERM = 11, 13

RMAX = 22.8                       # truncation of the Plummer spheres, structural units
HENON = 3.0 * math.pi / 16.0      # structural length in Henon units
LEVEL_SPLIT = 5                   # the reference driver's
# the arrays of a tree whose lengths depend on the particles
TREE = dict(groups=(BUF_GROUPS, 2, "<i4"), cells=(BUF_CELLS, 4, "<i4"), size=(BUF_SIZE, 4, "<f4"),
            mono=(BUF_MONO, 4, "<f4"), quad0=(BUF_QUAD0, 4, "<f4"), quad1=(BUF_QUAD1, 2, "<f4"))


def listed():
    return [
        # the smallest call: a star cluster of a thousand bodies
        dict(name="force_1k", kind="force", ic="plummer", n=1024, theta=0.5, eps=0.01),
        # monopole-only cells, larger leaves and smaller groups, a size that fills no tile
        dict(name="force_10k_mono", kind="force", ic="plummer", n=10007, theta=0.5, eps=0.01,
             nleaf=32, ncrit=48, mono=True),
        # the benchmark's first configuration: Plummer sphere of 2^16, theta 0.4
        dict(name="force_64k", kind="force", ic="plummer", n=65536, theta=0.4, eps=0.01),
        # Treecode<double>
        dict(name="force_30k_fp64", kind="force", ic="plummer", n=30011, theta=0.5, eps=0.01,
             fp64=True),
        # clustered particles held on the GPU, odd size
        dict(name="device_1m_clustered", kind="device", ic="clustered", n=1000003, theta=0.5,
             eps=0.002),
        # the build alone on the 20 million bodies of the reference's published build time
        dict(name="build_20m", kind="build", ic="plummer", n=20000000, theta=0.4, eps=0.002),
        # the plain walk at the size the metric is quoted at
        dict(name="device_16m", kind="device", ic="plummer", n=1 << 24, theta=0.4, eps=0.002),
        # the learned opening angle with its FP64 check, halo + disk
        dict(name="device_16m_learned", kind="device", ic="halo_disk", n=1 << 24, theta=0.4,
             eps=0.002, learned=True),
        # a small simulation: 8 steps and a snapshot
        dict(name="step_64k", kind="step", ic="plummer", n=65536, theta=0.5, eps=0.01, steps=8,
             dt=1.0 / 128),
        # the benchmark's second configuration with the learned angle: 8 steps and a snapshot
        dict(name="step_4m_learned", kind="step", ic="plummer", n=1 << 22, theta=0.5, eps=0.005,
             steps=8, dt=1.0 / 128, learned=True),
        # 256 independent systems of 2^10 to 2^16 bodies in one launch, captured steps
        dict(name="graph_ensemble", kind="graph", ic="plummer", systems=256, lo=10, hi=16,
             theta=0.5, eps=0.01, steps=8, dt=1.0 / 256),
        # training of the opening-angle network (forward, backward, Adam)
        dict(name="train_256", kind="train", samples=131072, batch=8192, steps=256),
    ]


def _log2(rng, lo, hi):
    """A whole number spread evenly over its logarithm, odd ones among them."""
    return max(2, int(round(2.0 ** rng.uniform(lo, hi))))


def draw(rng):
    kind = rng.choice(["force", "force", "device", "device", "build", "step", "graph", "train"])
    theta = rng.choice([0.4, 0.5, 0.5, 0.6, 0.75])
    eps = rng.choice([0.002, 0.005, 0.01])
    if kind == "train":
        return dict(kind=kind, samples=_log2(rng, 14, 18), batch=rng.choice([2048, 4096, 8192]),
                    steps=rng.randrange(64, 257))
    if kind == "graph":
        return dict(kind=kind, ic="plummer", systems=rng.randrange(16, 257), lo=10,
                    hi=rng.choice([12, 14, 16]), theta=rng.choice([0.5, 0.6]), eps=eps,
                    steps=rng.randrange(2, 9), dt=1.0 / 256)
    case = dict(kind=kind, ic=rng.choice(["plummer", "plummer", "clustered", "halo_disk"]),
                theta=theta, eps=eps)
    if kind == "force":
        case.update(n=_log2(rng, 10, 17), nleaf=rng.choice([16, 16, 24, 32, 48, 64]),
                    ncrit=rng.choice([64, 64, 48, 32]))
        option = rng.choice(["", "", "mono", "fp64"])
        if option:
            case[option] = True
        if option == "fp64":
            case["n"] = min(case["n"], 40009)
    elif kind == "device":
        case.update(n=_log2(rng, 17, 23))
        if case["ic"] != "clustered" and rng.random() < 0.4:
            case.update(learned=True, theta=0.4, eps=0.005)
    elif kind == "build":
        case.update(n=_log2(rng, 18, 24), nleaf=rng.choice([16, 16, 32]))
    else:
        case.update(ic="plummer", n=_log2(rng, 12, 21), steps=rng.randrange(1, 9), dt=1.0 / 128)
    return case


# ---- particles ---------------------------------------------------------------------

def _unit(n, g, dev):
    """Isotropic directions."""
    z = 2.0 * torch.rand(n, generator=g, device=dev, dtype=torch.float64) - 1.0
    p = 2.0 * math.pi * torch.rand(n, generator=g, device=dev, dtype=torch.float64)
    s = torch.sqrt(1.0 - z * z)
    return torch.stack([s * torch.cos(p), s * torch.sin(p), z], 1)


def _plummer(n, g, dev):
    """Positions and velocities of a Plummer sphere of unit mass, Henon units."""
    def rnd():
        return torch.rand(n, generator=g, device=dev, dtype=torch.float64)
    mmax = RMAX ** 3 / (1.0 + RMAX ** 2) ** 1.5
    r = 1.0 / torch.sqrt((rnd() * mmax).clamp_min(1e-12) ** (-2.0 / 3.0) - 1.0)
    # speed / escape speed from the density q^2 (1 - q^2)^3.5, by its tabulated integral
    q = torch.linspace(0.0, 1.0, 4097, device=dev, dtype=torch.float64)
    c = torch.cumsum(q * q * (1.0 - q * q).clamp_min(0.0) ** 3.5, 0)
    c = c / c[-1]
    u = rnd()
    k = torch.searchsorted(c, u).clamp(1, 4096)
    f = (u - c[k - 1]) / (c[k] - c[k - 1]).clamp_min(1e-300)
    speed = (q[k - 1] + f * (q[k] - q[k - 1])) * math.sqrt(2.0) * (1.0 + r * r) ** -0.25
    x = _unit(n, g, dev) * (r * HENON)[:, None]
    v = _unit(n, g, dev) * (speed / math.sqrt(HENON))[:, None]
    return x, v


def _particles(ic, n, seed, dev="cuda"):
    """(pos, vel): (n, 4) float32 tensors of (x, y, z, m) and (vx, vy, vz, m)."""
    g = torch.Generator(device=dev).manual_seed(int(seed) * 1000003 + 17)
    x, v = _plummer(n, g, dev)
    if ic == "clustered":     # 64 spheres, masses over three decades, in a box of half size 10
        m = torch.exp(math.log(1e-3) * torch.rand(64, generator=g, device=dev,
                                                  dtype=torch.float64))
        m = m / m.sum()
        centre = 10.0 * (2.0 * torch.rand(64, 3, generator=g, device=dev,
                                          dtype=torch.float64) - 1.0)
        at = (torch.arange(n, device=dev, dtype=torch.float64) + 0.5) / n
        own = torch.searchsorted(torch.cumsum(m, 0), at).clamp(0, 63)
        a = 0.5 * m[own] ** (1.0 / 3.0)
        x = centre[own] + x * a[:, None]
        v = v * torch.sqrt(m[own] / a)[:, None]
    elif ic == "halo_disk":   # a sphere of mass 0.8 and an exponential disk of mass 0.2
        nh = int(round(0.8 * n))
        v = v * math.sqrt(0.8)
        k, rd = n - nh, 0.3
        u = torch.rand(3, k, generator=g, device=dev, dtype=torch.float64).clamp_min(1e-12)
        r = (-rd * torch.log(u[0] * u[1])).clamp_max(10.0 * rd)
        p = 2.0 * math.pi * u[2]
        z = 0.03 * torch.atanh((2.0 * torch.rand(k, generator=g, device=dev,
                                                 dtype=torch.float64) - 1.0).clamp(-0.999999,
                                                                                   0.999999))
        x[nh:] = torch.stack([r * torch.cos(p), r * torch.sin(p), z], 1)
        inside = 0.8 * (r * r / (r * r + HENON * HENON)) ** 1.5
        inside += 0.2 * (1.0 - (1.0 + r / rd) * torch.exp(-r / rd))
        speed = torch.sqrt(inside / r)
        v[nh:] = torch.stack([-speed * torch.sin(p), speed * torch.cos(p), 0.0 * z], 1)
    x = x - x.mean(0)
    v = v - v.mean(0)
    mass = torch.full((n, 1), 1.0 / n, device=dev, dtype=torch.float64)
    return torch.cat([x, mass], 1).float(), torch.cat([v, mass], 1).float()


def _system_sizes(case):
    """Sizes of an ensemble's systems, even over their logarithm, large and small mixed."""
    k, lo, hi = case["systems"], case["lo"], case["hi"]
    order = sorted(range(k), key=lambda i: (i * 89) % k * k + i)
    return [int(round(2.0 ** (lo + (hi - lo) * (i + 0.5) / k))) for i in order]


def _case_particles(case, seed, dev="cuda"):
    if case["kind"] != "graph":
        return _particles(case["ic"], case["n"], seed, dev)
    sizes = _system_sizes(case)
    both = [_particles(case["ic"], nk, seed * 4099 + k, dev) for k, nk in enumerate(sizes)]
    return torch.cat([p for p, _ in both]), torch.cat([v for _, v in both])


# ---- training pairs ------------------------------------------------------------------

def _pairs(n, seed):
    """Feature rows and targets with the ranges of the pairs a walk collects: the
    eight features of a (group, cell) pair of random geometry, and a smooth
    target with scatter."""
    rng = np.random.default_rng(seed + 31)
    d = np.exp(rng.uniform(math.log(0.02), math.log(8.0), n))
    cell = d * np.exp(rng.uniform(math.log(0.1), math.log(1.2), n))
    rg = np.exp(rng.uniform(math.log(0.01), math.log(0.5), n))
    mass = np.clip((cell / 4.0) ** 2.2 * np.exp(rng.normal(0.0, 0.5, n)), 1e-7, 1.0)
    qn = 0.12 * np.exp(rng.normal(0.0, 0.4, n))
    cz, ck = rng.uniform(0.0, 1.0, n), rng.uniform(0.0, 1.0, n)
    x = np.stack([rg / (rg + d), rng.integers(20, 65, n) / 64.0, cell / (cell + d), d / (d + 32.0),
                  mass, qn / (1.0 + qn), cz, np.sqrt(1.0 - cz * cz) * ck], 1)
    y = (np.log2(cell / d) - np.log2(mass * (qn + 0.05) / d ** 2 + 1e-7) / 3.0 + 0.3 * x[:, 0]
         + 0.2 * cz + rng.normal(0.0, 0.3, n))
    return np.ascontiguousarray(x, np.float32), np.ascontiguousarray(y, np.float32)


# ---- preparing and running -------------------------------------------------------------

class _View:
    """A device array of a context, for torch; the tensor keeps the view, and the
    view the context that owns the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr=typestr,
                                             strides=None, version=2)


def _buffer(t, which, width, typestr):
    """The context's device array `which` as a tensor of `width` values a row."""
    ptr = ctypes.c_void_p()
    count = ctypes.c_int64()
    rc = bt.lib().bt_get_device_buffer(t._h, which, ctypes.byref(ptr), ctypes.byref(count))
    if rc != 0:
        raise RuntimeError("bt_get_device_buffer failed (%d)" % rc)
    return torch.as_tensor(_View(t, ptr.value, (count.value, width), typestr), device="cuda")


def _context(case):
    t = bt.Treecode(case["eps"], case["theta"], case.get("ncrit", 64), fp64=case.get("fp64", False))
    if case["kind"] == "graph":
        off = np.concatenate([[0], np.cumsum(_system_sizes(case))]).astype(np.int32)
        t.alloc(int(off[-1]), off)
    else:
        t.alloc(case["n"])
    if case.get("mono"):
        t.set_quadrupole(False)
    if case.get("learned"):
        t.use_learned_theta()
    return t


def _evaluate(t, case):
    """The reference's sequence of phases."""
    t.buildTree(case.get("nleaf", 16))
    t.computeMultipoles()
    t.makeGroups(LEVEL_SPLIT, case.get("ncrit", 64))
    t.computeForces()


def prepare(case, seed):
    s = dict(case=case)
    if case["kind"] == "train":
        s["x"], s["y"] = _pairs(case["samples"], seed)
        t = s["t"] = bt.Treecode(0.01, 0.5, 64)
        t.mlp_init(seed + 1, float(np.mean(s["y"])))
        s["p0"] = t.mlp_params()
        return s
    pos, vel = _case_particles(case, seed)
    t = s["t"] = _context(case)
    if case["kind"] in ("device", "build"):
        s["pos"], s["vel"] = pos, vel
        if case["kind"] == "build":   # room for the tree: a cell for every two particles
            rows = case["n"] // 2 + 4096
            s["tree"] = {name: torch.zeros(rows, width, device="cuda",
                                           dtype=torch.int32 if typestr == "<i4" else torch.float32)
                         for name, (_, width, typestr) in TREE.items()}
        torch.cuda.synchronize()
        return s
    real = np.float64 if case.get("fp64") else np.float32
    s["pos"], s["vel"] = pos.cpu().numpy().astype(real), vel.cpu().numpy().astype(real)
    if case["kind"] in ("step", "graph"):     # a run under way: its forces are current
        t.ptcl_h2d(s["pos"], s["vel"])
        _evaluate(t, case)
    return s


def run(state):
    case, t = state["case"], state["t"]
    kind = case["kind"]
    if kind == "train":
        t.set_mlp_params(state["p0"])
        curve = t.mlp_train(state["x"], state["y"], steps=case["steps"], batch=case["batch"])
        return dict(params=t.mlp_params(), loss=curve)
    if kind == "force":
        t.ptcl_h2d(state["pos"], state["vel"])
        _evaluate(t, case)
        return dict(acc=t.acc(bt.ORDER_INPUT))
    if kind in ("step", "graph"):
        if kind == "graph":
            t.step_graph(case["dt"], 16, LEVEL_SPLIT, 64, nsteps=case["steps"])
        else:
            for _ in range(case["steps"]):
                t.step(case["dt"], 16, LEVEL_SPLIT, 64)
        pos, vel = t.ptcl_d2h(bt.ORDER_INPUT)
        return dict(pos=pos, vel=vel)
    rc = bt.lib().bt_set_particles_device(t._h, ctypes.c_void_p(state["pos"].data_ptr()),
                                          ctypes.c_void_p(state["vel"].data_ptr()))
    if rc != 0:
        raise RuntimeError("bt_set_particles_device failed (%d)" % rc)
    if kind == "device":
        _evaluate(t, case)
        return dict(acc=_buffer(t, BUF_ACC, 4, "<f4"), perm=_buffer(t, BUF_PERM, 1, "<i4"))
    t.buildTree(case.get("nleaf", 16))
    t.computeMultipoles()
    t.makeGroups(LEVEL_SPLIT, 64)
    for name, (which, width, typestr) in TREE.items():
        got = _buffer(t, which, width, typestr)
        state["tree"][name][:len(got)].copy_(got)
    torch.cuda.current_stream().synchronize()   # the context's arrays are free again
    return dict(state["tree"], pos=_buffer(t, BUF_POS, 4, "<f4"),
                perm=_buffer(t, BUF_PERM, 1, "<i4"), levels=_buffer(t, BUF_LEVELS, 2, "<i4"))


# ---- work and exact results ------------------------------------------------------------

def _walk_flops(n, theta, learned=False):
    """Flops of one walk over n particles, 20 a particle pair and 64 a cell: a fit
    to measured walks (they grow with the logarithm of n and about as theta^-1.9;
    the learned angle does a quarter of theta = 0.4's), at most the direct sum's."""
    per = 21.5e3 * (0.4 / theta) ** 1.9 * max(1.0, math.log2(n) - 6.3)
    return n * min(20.0 * n, per * (0.25 if learned else 1.0))


def work(case):
    if case["kind"] == "train":
        # forward and backward products of 1344 weights, three multiply-adds each
        return dict(bytes=36.0 * case["samples"],
                    flops=6.0 * 1344 * case["batch"] * float(case["steps"]))
    sizes = _system_sizes(case) if case["kind"] == "graph" else [case["n"]]
    n = sum(sizes)
    b = 8.0 if case.get("fp64") else 4.0
    learned = case.get("learned", False)
    flops = sum(_walk_flops(k, case["theta"], learned) for k in sizes)
    if learned:
        flops += 18.0 * 256 * n           # the FP64 check of 256 targets
    if case["kind"] in ("step", "graph"):
        # each step reads and writes the particles and their accelerations
        return dict(bytes=case["steps"] * n * 20 * b, flops=case["steps"] * flops)
    if case["kind"] == "build":
        cells = 0.24 * n * 16 / case.get("nleaf", 16)
        return dict(bytes=n * (8 * b + 4 * b + 4) + cells * 2 * (16 + 14 * b), flops=0.0)
    return dict(bytes=n * (8 * b + 4 * b), flops=flops)


def _direct(pos, eps, offsets):
    """(ax, ay, az, phi) in FP64 by direct summation within each system; phi has the
    self term -m/eps, as the walk's."""
    out = torch.zeros(len(pos), 4, device=pos.device, dtype=torch.float64)
    for b, e in zip(offsets[:-1], offsets[1:]):
        src = pos[b:e]
        sx, sy, sz, sm = (src[:, k].contiguous() for k in range(4))
        rows = max(1, (1 << 26) // len(src))
        for i in range(b, e, rows):
            p = pos[i:min(e, i + rows)]
            dx, dy, dz = (s[None] - p[:, k:k + 1] for k, s in enumerate((sx, sy, sz)))
            r = torch.rsqrt(dx * dx + dy * dy + dz * dz + eps * eps)
            w = sm[None] * r
            out[i:i + len(p), 3] = -w.sum(1)
            w = w * r * r
            for k, d in enumerate((dx, dy, dz)):
                out[i:i + len(p), k] = (w * d).sum(1)
    return out


def exact(case, seed):
    kind = case["kind"]
    # the network is FP16 by definition, and the order of the tree's particles and
    # cells follows from its float keys: neither has a 64-bit value of its own
    if kind not in ("force", "step", "graph"):
        return None
    sizes = _system_sizes(case) if kind == "graph" else [case["n"]]
    if sum(float(k) * k for k in sizes) * (1 + case.get("steps", 0)) > 8e10:
        return None
    offsets = np.concatenate([[0], np.cumsum(sizes)]).tolist()
    pos, vel = (v.double() for v in _case_particles(case, seed))
    eps = float(case["eps"]) if case.get("fp64") else float(np.float32(case["eps"]))
    acc = _direct(pos, eps, offsets)
    if kind == "force":
        return dict(acc=acc)
    dt = float(np.float32(case["dt"]))
    for _ in range(case["steps"]):
        vel[:, :3] += acc[:, :3] * (0.5 * dt)
        pos[:, :3] += vel[:, :3] * dt
        acc = _direct(pos, eps, offsets)
        vel[:, :3] += acc[:, :3] * (0.5 * dt)
    return dict(pos=pos, vel=vel)
