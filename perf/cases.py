"""Performance cases of the gravity path, through its public entry points.

A case is one call (or one short sequence of calls) that a program built on
this package makes:

* ``step``     -- a torch program that owns its particles hands the new
  positions over (``Driver.load_device``) and asks for the forces
  (``Driver.compute_forces``), once per step of its own integrator;
* ``force``    -- one force evaluation of particles that stay in the context;
* ``run``      -- ``Driver.run``: a block of kick-drift steps from a given state;
* ``lists``    -- the stage calls of ``Driver::run`` one by one, ending in
  ``start_down`` (traversal lists, then the visitor calls over them);
* ``vjp``      -- the vector-Jacobian product of one force evaluation;
* ``train``    -- ``autograd.trajectory`` with a loss and its backward pass.

Sizes, bucket sizes, opening angles and softenings are those of the benchmark
(100k and 1M Plummer spheres, the 16M halo mixture, the 256k adjoint), of the
tests and of the 30k-particle sample the reference ships, plus odd sizes
between them.

Results that the compensated-FP32 form computes are returned as float32, the
precision its arithmetic carries; FP64 results are returned as the float64
arrays of the context.
"""
import ctypes
import itertools
import math

import torch

from paratreet_amd import _lib
from paratreet_amd import autograd as _ag
from paratreet_amd.gravity import PT_FP32C, PT_FP64, Configuration, Driver, GravityVisitor

_DEFAULTS = {"kind": "force", "dist": "plummer", "precision": "fp64", "bucket": 16, "theta": 0.7,
             "eps": 0.01, "hexadecapole": False, "replicas": -1, "steps": 0}


def listed():
    return [
        # the smallest sets, forces every step of the caller's own integrator:
        # launches and latency are all there is
        _case("step_1k_fp64", kind="step", n=1000, bucket=12),
        # the size of the reference's sample file with its two softenings
        # (gas and dark particles), the application's default bucket of 12
        _case("step_30k_gasdark_fp64", kind="step", dist="gasdark", n=30000, bucket=12),
        # the 100k benchmark workload
        _case("force_100k_fp32c", n=100000, bucket=12, precision="fp32c"),
        # the headline benchmark workload
        _case("force_1m_fp32c", n=1000000, eps=0.005, precision="fp32c"),
        # the same physics in plain FP64 at an odd size
        _case("force_777k_fp64", n=777777, eps=0.005),
        # the largest benchmark workload: 64 halos on a uniform background
        _case("force_16m_halo_fp32c", dist="halo", n=16000000, bucket=32, precision="fp32c"),
        # the reference's default build (moments to fourth order)
        _case("hexa_1m_fp32c", n=1000000, eps=0.005, precision="fp32c", hexadecapole=True),
        # a periodic box: 27 replicas and the Ewald correction
        _case("periodic_50k_fp64", dist="box", n=50000, bucket=12, eps=0.002, replicas=1),
        # the stage-by-stage calls with lists kept
        _case("lists_200k_fp64", kind="lists", n=200003, bucket=12),
        # a block of steps of a small simulation
        _case("run_20k_10steps_fp64", kind="run", n=20011, bucket=12, steps=10),
        # the differentiable force at the 256k adjoint workload's size
        _case("vjp_256k_fp64", kind="vjp", n=262144, eps=0.005),
        # one optimisation step through a short trajectory, halo mixture
        _case("train_64k_4steps_fp32c", kind="train", dist="halo", n=65536, bucket=32, steps=4,
              precision="fp32c"),
    ]


def draw(rng):
    """One more case of the ranges above (a pass costs less than the 16M one)."""
    kind = rng.choice(["step", "step", "force", "force", "force", "hexa", "periodic", "run",
                       "lists", "vjp", "train"])
    c = {"precision": rng.choice(["fp64", "fp32c"]), "bucket": rng.choice([7, 8, 12, 16, 24, 32]),
         "theta": round(rng.uniform(0.55, 0.9), 3), "dist": rng.choice(["plummer", "halo", "gasdark"]),
         "eps": round(10 ** rng.uniform(-2.6, -1.7), 6)}
    lo, hi = {"step": (600, 200000), "force": (3000, 2500000), "hexa": (3000, 1000000),
              "periodic": (1000, 60000), "run": (1000, 100000), "lists": (1000, 300000),
              "vjp": (1000, 200000), "train": (1000, 60000)}[kind]
    c["n"] = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    c["kind"] = kind if kind not in ("hexa", "periodic") else "force"
    if kind == "hexa":
        c["hexadecapole"] = True
    if kind == "periodic":
        c.update(dist="box", replicas=1, eps=0.002)
    if kind == "run":
        c["steps"] = rng.randint(3, 10)
    if kind == "train":
        c["steps"] = rng.randint(2, 4)
    return {**_DEFAULTS, **c}


def _case(name, **kw):
    return {"name": name, **_DEFAULTS, **kw}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

_DT = 1e-3


def _isotropic(n, g):
    cz = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    ph = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (2 * math.pi)
    sz = (1 - cz * cz).sqrt()
    return torch.stack([sz * ph.cos(), sz * ph.sin(), cz], 1)


def _plummer(n, g, rmax=10.0):
    """Plummer sphere, G = M = a = 1, radii to rmax, isotropic velocities from
    the distribution function q^2 (1 - q^2)^(7/2) (inverse of its table)."""
    top = (1 + rmax ** -2) ** -1.5
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (top - 1e-9) + 1e-9
    r = (u ** (-2.0 / 3.0) - 1).rsqrt()
    q = torch.linspace(0, 1, 4097, dtype=torch.float64, device="cuda")
    cdf = torch.cumsum(q * q * (1 - q * q) ** 3.5, 0)
    v = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    q = q[torch.searchsorted(cdf / cdf[-1], v).clamp(max=4096)]
    pos = _isotropic(n, g) * r[:, None]
    vel = _isotropic(n, g) * (q * math.sqrt(2.0) * (1 + r * r) ** -0.25)[:, None]
    return pos, vel


def _inputs(case, seed):
    """(pos, vel, mass, soft) on the GPU, from the seed alone."""
    n, eps = case["n"], case["eps"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    mass = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    soft = torch.full((n,), eps, dtype=torch.float64, device="cuda")
    if case["dist"] == "plummer":
        pos, vel = _plummer(n, g)
    elif case["dist"] == "gasdark":
        # a tenth of the particles are light and widely softened
        pos, vel = _plummer(n, g)
        gas = torch.rand(n, generator=g, device="cuda") < 0.1
        soft = torch.where(gas, 20 * soft, 0.4 * soft)
        mass = torch.where(gas, 0.2 * mass, 1.1 * mass)
    elif case["dist"] == "halo":
        # log-normal halos with centres in a cube and a 20% background
        halos = 64 if n >= 1000000 else 16
        hm = torch.randn(halos, generator=g, device="cuda", dtype=torch.float64).exp()
        which = torch.searchsorted(
            torch.cumsum(hm / hm.sum(), 0),
            torch.rand(n, generator=g, device="cuda", dtype=torch.float64)).clamp(max=halos - 1)
        centre = torch.rand(halos, 3, generator=g, device="cuda", dtype=torch.float64) * 100
        scale = (hm / hm.mean()) ** (1.0 / 3.0)
        pos, vel = _plummer(n, g)
        pos = centre[which] + pos * scale[which, None]
        vel = vel * (hm / hm.sum() / scale).sqrt()[which, None]
        back = torch.rand(n, generator=g, device="cuda") < 0.2
        uni = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64) * 100
        pos = torch.where(back[:, None], uni, pos)
        vel = torch.where(back[:, None], torch.zeros_like(vel), vel)
    else:  # "box": clumps and a uniform half in the unit box
        uni = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64)
        centre = torch.rand(8, 3, generator=g, device="cuda", dtype=torch.float64)
        k = torch.randint(0, 8, (n,), generator=g, device="cuda")
        clump = centre[k] + 0.03 * torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float64)
        half = torch.rand(n, generator=g, device="cuda") < 0.5
        pos = torch.where(half[:, None], uni, clump - clump.floor())
        vel = torch.zeros_like(pos)
    assert all(t.dtype == torch.float64 for t in (pos, vel, mass, soft))
    return pos, vel, mass, soft


class _View:
    """A device array of a context, as torch reads foreign device memory; the
    tensor made from it holds this object, and so the context that owns the
    memory."""

    def __init__(self, driver, ptr, n):
        self.driver = driver
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False),
                                         "version": 3}


def _tensor(driver, ptr, n):
    return torch.as_tensor(_View(driver, ptr, n), device="cuda")


def prepare(case, seed):
    case = {**_DEFAULTS, **case}
    pos, vel, mass, soft = _inputs(case, seed)
    cfg = Configuration(max_particles_per_leaf=case["bucket"])
    if case["hexadecapole"]:
        cfg.hexadecapole = True
    if case["replicas"] >= 0:
        cfg.periodic, cfg.fPeriod, cfg.nReplicas = 1, (1.0, 1.0, 1.0), case["replicas"]
    s = {"case": case, "driver": Driver(cfg), "mass": mass, "soft": soft,
         "precision": PT_FP32C if case["precision"] == "fp32c" else PT_FP64,
         "x": pos.t().contiguous(), "v": vel.t().contiguous()}
    if case["kind"] == "train":
        s["x0"], s["v0"], s["m0"] = (t.clone().requires_grad_() for t in (pos, vel, mass))
    if case["kind"] == "vjp":
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        s["w"] = torch.randn(case["n"], 3, generator=g, device="cuda", dtype=torch.float64)
        s["gx"], s["gm"] = torch.empty_like(s["w"]), torch.empty_like(mass)
    torch.cuda.synchronize()
    _load(s)
    return s


def _load(s):
    x, v = s["x"], s["v"]
    s["driver"].load_device(s["case"]["n"], x[0].data_ptr(), x[1].data_ptr(), x[2].data_ptr(),
                            s["mass"].data_ptr(), s["soft"].data_ptr(), v[0].data_ptr(),
                            v[1].data_ptr(), v[2].data_ptr())


def _out(s, counters, *fields):
    """The context's result arrays (float32 copies in the FP32C form)."""
    view, n = s["driver"].device_view(), s["case"]["n"]
    got = [_tensor(s["driver"], getattr(view, f), n) for f in fields]
    if s["precision"] == PT_FP32C:
        got = [t.float() for t in got]
    return {"values": got, "counters": [int(c) for c in counters]}


def run(s):
    c, d = s["case"], s["driver"]
    kind, theta, prec = c["kind"], c["theta"], s["precision"]
    if kind in ("step", "force"):
        if kind == "step":
            _load(s)
        return _out(s, d.compute_forces(theta, prec), "ax", "ay", "az", "pot")
    if kind == "run":
        _load(s)
        cnt = d.run(c["steps"], _DT, theta, prec)
        return _out(s, cnt, "x", "y", "z", "vx", "vy", "vz")
    if kind == "lists":
        d.remake_universe()
        d.assign_keys()
        d.build_tree()
        cnt = d.start_down(GravityVisitor((0.0, 0.0, 0.0), theta), prec)
        return _out(s, cnt, "ax", "ay", "az", "pot")
    if kind == "vjp":
        d.set_adjoint_precision(prec)
        d._check(d.L.pt_force_vjp(d.ctx, theta, _lib.PT_FORCE_TREE,
                                  ctypes.c_void_p(s["w"].data_ptr()),
                                  ctypes.c_void_p(s["gx"].data_ptr()),
                                  ctypes.c_void_p(s["gm"].data_ptr()), _lib.PT_DEVICE))
        got = [s["gx"], s["gm"]]
    else:
        x0, v0, m = s["x0"], s["v0"], s["m0"]
        x0.grad = v0.grad = m.grad = None
        xt, vt = _ag.trajectory(x0, v0, m, s["soft"], steps=c["steps"], dt=_DT, theta=theta,
                                precision=c["precision"], driver=d)
        # kinetic energy and a pull towards the centre at the end of the path
        (m * ((vt * vt).sum(1) + (xt * xt).sum(1))).sum().backward()
        got = [xt.detach(), vt.detach(), x0.grad, v0.grad, m.grad]
    return {"values": [t.float() for t in got] if prec == PT_FP32C else got}


def work(case):
    """Each particle's inputs read once and its results written once; 20
    flops per particle pair and 67 per particle and closed node (the counts
    of the benchmark), with the pair counts of these tree parameters per
    particle fitted on counted runs; the adjoint of a pair at 2.5 times it."""
    case = {**_DEFAULTS, **case}
    n, b, th = case["n"], case["bucket"], case["theta"]
    reach = (0.7 / th) ** 2.2 * min(1.0, math.log10(n) / 6.0)
    pp, pc = 85.0 * b * reach, 950.0 * (16.0 / b) ** 0.3 * reach
    flops = n * (20.0 * min(pp, n) + (200.0 if case["hexadecapole"] else 67.0) * min(pc, n))
    nbytes = n * 72.0
    if case["replicas"] >= 0:
        flops *= 2.0
        flops += n * 150 * 40.0
    if case["kind"] == "run":
        flops, nbytes = flops * case["steps"], nbytes * case["steps"]
    if case["kind"] == "vjp":
        flops, nbytes = 2.5 * flops, n * 96.0
    if case["kind"] == "train":
        flops, nbytes = 3.5 * flops * case["steps"], n * 232.0 * case["steps"]
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same results in plain torch, FP64
# ---------------------------------------------------------------------------

_LEAF, _INTERNAL = 1, 2
_MAX_DEPTH = 21
_PAIRS = 1 << 23  # pairs evaluated at once


class _Tree:
    """Octree over Morton keys: the reference's split rule, nodes in level
    order, particles in key order (ties by index)."""

    def __init__(self, x, bucket):
        lo, hi = x.amin(0), x.amax(0)
        half = (1.0 + 1.91e-6) * 0.5 * (hi - lo).max()
        mid = (lo + hi) / 2.0
        lo, hi = mid - half, mid + half
        q = torch.floor((x - lo) / (hi - lo) * 2097152.0).clamp(0, 2097151).long()
        key = torch.zeros(len(x), dtype=torch.int64, device=x.device)
        for b in range(_MAX_DEPTH):
            for a in range(3):
                key |= ((q[:, a] >> b) & 1) << (3 * b + 2 - a)
        key, self.perm = torch.sort(key, stable=True)
        dev = x.device
        prefix = torch.zeros(1, dtype=torch.int64, device=dev)
        begin, count = prefix.clone(), prefix + len(x)
        levels, base = [], 0
        for d in range(_MAX_DEPTH + 1):
            split = (count > bucket) & (d < _MAX_DEPTH)
            kind = torch.where(split, _INTERNAL, (count > 0).long() * _LEAF)
            first = torch.full_like(begin, -1)
            first[split] = base + len(begin) + 8 * torch.arange(int(split.sum()), device=dev)
            levels.append((begin, count, kind, first))
            if not bool(split.any()):
                break
            base += len(begin)
            end = (begin + count)[split]
            prefix = (prefix[split, None] * 8 + torch.arange(8, device=dev)).reshape(-1)
            shift = 3 * (_MAX_DEPTH - d - 1)
            begin = torch.searchsorted(key, prefix << shift)
            stop = torch.cat([begin[1:], begin[-1:]])
            stop[7::8] = end
            count = stop - begin
        self.begin, self.count, self.kind, self.first = (torch.cat(t) for t in zip(*levels))
        leaves = torch.nonzero(self.kind == _LEAF)[:, 0]
        self.buckets = leaves[torch.argsort(self.begin[leaves])]
        # every node's particles, node after node
        self.pid = _ranges(self.begin, self.begin, self.count)[1]


def _ranges(ids, begin, count):
    """(id, index) for every index in each id's range."""
    rep = torch.repeat_interleave(torch.arange(len(ids), device=ids.device), count)
    start = torch.cumsum(count, 0) - count
    return ids[rep], torch.arange(len(rep), device=ids.device) - start[rep] + begin[rep]


_Q = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]


def _moments(t, x, m, e):
    """Differentiable node moments: mass, centre, second moments, softening."""
    pid, count = t.pid, t.count
    mp = m[pid]
    mass = _long_sums(mp, count)
    safe = torch.where(mass > 0, mass, 1.0)
    cm = _long_sums(mp[:, None] * x[pid], count) / safe[:, None]
    u = x[pid] - cm.repeat_interleave(count, 0)
    q = _long_sums(torch.stack([mp * u[:, i] * u[:, j] for i, j in _Q], 1), count)
    return {"mass": mass, "cm": cm, "q": q, "soft": _long_sums(mp * e[pid], count) / safe}


def _exponents(order):
    return [(a, b, order - a - b) for a in range(order, -1, -1) for b in range(order - a, -1, -1)]


def _high_moments(t, x, m, cm):
    """Raw third and fourth moments about the centre, by exponents."""
    u = (x[t.pid] - cm.repeat_interleave(t.count, 0)).t()
    return {ex: _long_sums(m[t.pid] * u[0] ** ex[0] * u[1] ** ex[1] * u[2] ** ex[2], t.count)
            for order in (3, 4) for ex in _exponents(order)}


def _boxes(t, x):
    return (_long_sums(x[t.pid], t.count, "min", math.inf),
            _long_sums(x[t.pid], t.count, "max", -math.inf))


def _box_dsq(lo, hi, p):
    d = torch.maximum(torch.clamp(lo - p, min=0), torch.clamp(p - hi, min=0))
    return (d * d).sum(1)


def _spline(r2, twoh):
    """GravityVisitor::SPLINE's force factor."""
    r = r2.sqrt()
    h = 2.0 / twoh
    u = r * h
    inner = h ** 3 * (4.0 / 3.0 - 1.2 * u * u + 0.5 * u ** 3)
    outer = -1.0 / 15.0 / r ** 3 + h ** 3 * (8.0 / 3.0 - 3.0 * u + 1.2 * u * u - u ** 3 / 6.0)
    return torch.where(r < twoh, torch.where(u < 1.0, inner, outer), 1.0 / (r * r2))


def _splineq(r2, twoh):
    """GravityVisitor::SPLINEQ's four factors, grouped as the reference has them."""
    dir = r2.rsqrt()
    h = 2.0 / twoh
    u = h / dir
    inner = (h * 1.4 - 2.0 / 3.0 * u ** 2 + 0.3 * u ** 4 - 0.1 * u ** 5,
             h ** 3 * 4.0 / 3.0 - 1.2 * u ** 2 + 0.5 * u ** 3,
             h ** 5 * 2.4 - 1.5 * u, 1.5 * h ** 6 * dir)
    outer = (-dir / 15.0 + h * 1.6 - 4.0 / 3.0 * u ** 2 + u ** 3 - 0.3 * u ** 4 + u ** 5 / 30.0,
             -dir ** 3 / 15.0 + h ** 3 * 8.0 / 3.0 - 3.0 * u + 1.2 * u ** 2 - u ** 3 / 6.0,
             -0.2 * dir ** 5 + 3.0 * h ** 4 * dir - 2.4 * h ** 5 + 0.5 * u,
             -dir ** 7 + 3.0 * h ** 4 * dir ** 3 - 0.5 * h ** 6 * dir)
    far = (dir, dir ** 3, 3.0 * dir ** 5, 15.0 * dir ** 7)
    near, first = r2 < twoh * twoh, u < 1.0
    return [torch.where(near, torch.where(first, i, o), f) for i, o, f in zip(inner, outer, far)]


def _pair_leaf(xt, et, xs, ms, es):
    d = xs - xt
    r2 = (d * d).sum(1)
    own = r2 == 0
    f = torch.where(own, 0.0, ms * _spline(torch.where(own, 1.0, r2), es + et))
    return d * f[:, None], None


def _pair_node(mono, xt, et, cm, mass, q, soft):
    r = xt - cm
    r2 = (r * r).sum(1)
    a, b, c, d = _splineq(r2, soft + et)
    qr = torch.stack([q[:, 0] * r[:, 0] + q[:, 1] * r[:, 1] + q[:, 2] * r[:, 2],
                      q[:, 1] * r[:, 0] + q[:, 3] * r[:, 1] + q[:, 4] * r[:, 2],
                      q[:, 2] * r[:, 0] + q[:, 4] * r[:, 1] + q[:, 5] * r[:, 2]], 1)
    half = 0.5 * (qr * r).sum(1)
    tr = 0.5 * (q[:, 0] + q[:, 3] + q[:, 5])
    radial = b * mass + d * half - c * tr
    acc = c[:, None] * qr - radial[:, None] * r
    pot = b * tr - mass * a - c * half
    alone = -(mass * r2.rsqrt() / r2)[:, None] * r
    return torch.where(mono[:, None], alone, acc), torch.where(mono, 0.0, pot)


def _pair_node_hexa(mono, xt, cm, mass, q, high):
    """Multipoles to fourth order; the force is minus the potential's gradient."""
    with torch.enable_grad():
        r = (xt - cm).requires_grad_()
        x, y, z = r[:, 0], r[:, 1], r[:, 2]
        r2 = (r * r).sum(1)
        p = [x, y, z]
        a2 = sum((1 if i == j else 2) * q[:, k] * p[i] * p[j] for k, (i, j) in enumerate(_Q))
        t2 = q[:, 0] + q[:, 3] + q[:, 5]

        def contract(order, comp):
            tot = 0.0
            for a, b, c in _exponents(order):
                mult = math.factorial(order) // (math.factorial(a) * math.factorial(b) * math.factorial(c))
                tot = tot + mult * comp(a, b, c) * x ** a * y ** b * z ** c
            return tot

        def trace(a, b, c):
            return high[(a + 2, b, c)] + high[(a, b + 2, c)] + high[(a, b, c + 2)]

        a3, a4 = (contract(o, lambda a, b, c: high[(a, b, c)]) for o in (3, 4))
        t3, t4 = contract(1, trace), contract(2, trace)
        t44 = trace(2, 0, 0) + trace(0, 2, 0) + trace(0, 0, 2)
        ir = r2.rsqrt()
        pot = -(mass * ir + 0.5 * (3 * a2 - t2 * r2) * ir ** 5 + 0.5 * (5 * a3 - 3 * r2 * t3) * ir ** 7
                + 0.125 * (35 * a4 - 30 * r2 * t4 + 3 * r2 * r2 * t44) * ir ** 9)
        acc = -torch.autograd.grad(pot.sum(), r)[0]
    alone = -(mass * r2.rsqrt() / r2).detach()[:, None] * r.detach()
    return torch.where(mono[:, None], alone, acc), torch.where(mono, 0.0, pot.detach())


class _Field:
    """The tree's force on particles in key order, and its adjoint."""

    def __init__(self, case, x, m, e):
        self.case, self.tree = case, _Tree(x, case["bucket"])
        t = self.tree
        self.x, self.m, self.e = x[t.perm], m[t.perm], e[t.perm]
        self.node = _moments(t, self.x, self.m, self.e)
        self.lo, self.hi = _boxes(t, self.x)
        cm = self.node["cm"]
        self.high = _high_moments(t, self.x, self.m, cm) if case["hexadecapole"] else None
        corner = torch.maximum(cm - self.lo, self.hi - cm)
        radius = torch.where(t.kind == _INTERNAL, (corner * corner).sum(1).sqrt(),
                             0.5 * ((self.hi - self.lo) ** 2).sum(1).sqrt())
        self.radius = torch.where(t.count > 1, radius, 1.0)

    def opened(self, bk, nd, off):
        """GravityVisitor::open for (bucket node, node) pairs."""
        th, cm = self.case["theta"], self.node["cm"][nd] + off
        few = self.tree.count[nd] <= 6
        dsq = _box_dsq(self.lo[bk], self.hi[bk], cm)
        op = few | (dsq <= self.radius[nd] ** 2 * (4.0 / 3.0 / (th * th)))
        if self.high is not None:
            at = self.node["cm"][bk] + off
            sb, sn = 2.0 * self.node["soft"][bk], 2.0 * self.node["soft"][nd]
            meet = ((at - self.node["cm"][nd]) ** 2).sum(1) <= (sb + sn) ** 2
            meet |= _box_dsq(self.lo[nd], self.hi[nd], at) <= sb * sb
            op |= meet & (dsq <= (self.radius[nd] * math.sqrt(4.0 / 3.0) / th ** 4) ** 2)
        return op

    def monopole(self, bk, nd, off):
        """GravityVisitor::openSoftening."""
        cm, sn = self.node["cm"][nd] + off, 2.0 * self.node["soft"][nd]
        meet = ((cm - self.node["cm"][bk]) ** 2).sum(1) <= (sn + 2.0 * self.node["soft"][bk]) ** 2
        return meet | (_box_dsq(self.lo[bk], self.hi[bk], cm) <= sn * sn)

    def pairs(self, off, counters):
        """Parts of the interaction list, targets in order: (kind, targets,
        entries per target, sources, monopole), with a row of the last two
        per entry: source particles ("leaf") or nodes ("node")."""
        t = self.tree
        for bks in torch.split(t.buckets, 2048):
            bk, nd = torch.arange(len(bks), device=bks.device), torch.zeros_like(bks)
            owner, tg = _ranges(bk, t.begin[bks], t.count[bks])
            while len(bk):
                leaf, inner = t.kind[nd] == _LEAF, t.kind[nd] == _INTERNAL
                row, src = _ranges(bk[leaf], t.begin[nd[leaf]], t.count[nd[leaf]])
                n_src = torch.bincount(row, minlength=len(bks))
                counters[1] += int((n_src * t.count[bks]).sum())
                yield from self._parts("leaf", tg, owner, n_src, src, None)
                bk, nd = bk[inner], nd[inner]
                op = self.opened(bks[bk], nd, off)
                row, src = bk[~op], nd[~op]
                n_src = torch.bincount(row, minlength=len(bks))
                counters[0] += int((n_src * t.count[bks]).sum())
                counters[2] += int(op.sum())
                counters[3] += len(src)
                yield from self._parts("node", tg, owner, n_src, src,
                                       self.monopole(bks[row], src, off))
                bk = bk[op].repeat_interleave(8)
                nd = (t.first[nd[op], None] + torch.arange(8, device=nd.device)).reshape(-1)

    @staticmethod
    def _parts(kind, tg, owner, n_src, src, mono):
        """Every target with its owner's sources, about _PAIRS rows at a time."""
        start = torch.cumsum(n_src, 0) - n_src
        count = n_src[owner]
        part = torch.cumsum(count, 0) // _PAIRS
        cuts = (torch.nonzero(part[1:] != part[:-1])[:, 0] + 1).tolist()
        for a, b in zip([0] + cuts, cuts + [len(tg)]):
            if int(count[a:b].sum()):
                _, row = _ranges(tg[a:b], start[owner[a:b]], count[a:b])
                yield kind, tg[a:b], count[a:b], src[row], None if mono is None else mono[row]

    def rows(self, kind, tg, count, sr, x, m, node):
        """The inputs of a part's pairs, a row each."""
        tg = tg.repeat_interleave(count)
        if kind == "leaf":
            return [x[tg], x[sr], m[sr]], (self.e[tg], self.e[sr])
        return ([x[tg], node["cm"][sr], node["mass"][sr], node["q"][sr], node["soft"][sr]],
                (self.e[tg], sr))

    def evaluate(self, kind, mono, off, rows, rest):
        if kind == "leaf":
            xt, xs, ms = rows
            return _pair_leaf(xt, rest[0], xs + off, ms, rest[1])
        xt, cm, mass, q, soft = rows
        if self.high is not None:
            return _pair_node_hexa(mono, xt, cm + off, mass, q,
                                   {k: v[rest[1]] for k, v in self.high.items()})
        return _pair_node(mono, xt, rest[0], cm + off, mass, q, soft)

    def force(self):
        """(acc, pot, counters), particles in input order."""
        n, r = len(self.x), max(self.case["replicas"], 0)
        acc, pot, counters = torch.zeros_like(self.x), torch.zeros_like(self.m), [0, 0, 0, 0]
        for rep in itertools.product(range(-r, r + 1), repeat=3):
            off = torch.tensor(rep, dtype=self.x.dtype, device=self.x.device)
            for kind, tg, count, sr, mono in self.pairs(off, counters):
                rows, rest = self.rows(kind, tg, count, sr, self.x, self.m, self.node)
                a, p = self.evaluate(kind, mono, off, rows, rest)
                acc[tg] += _sums(a, count)
                if p is not None:
                    pot[tg] += _sums(p, count)
        if self.case["replicas"] >= 0:
            a, p = _ewald(self.x, {k: v[0] for k, v in self.node.items()}, self.case["replicas"])
            acc, pot = acc + a, pot + p
        back = torch.empty_like(self.tree.perm)
        back[self.tree.perm] = torch.arange(n, device=back.device)
        return acc[back], pot[back], counters

    def vjp(self, w):
        """(da/dx)^T w and (da/dm)^T w, the interactions held fixed."""
        t = self.tree
        off = torch.zeros(3, dtype=self.x.dtype, device=self.x.device)
        gx, gm, ws = torch.zeros_like(self.x), torch.zeros_like(self.m), w[t.perm]
        gnode = {k: torch.zeros_like(v) for k, v in self.node.items()}
        for kind, tg, count, sr, mono in self.pairs(off, [0, 0, 0, 0]):
            rows, rest = self.rows(kind, tg, count, sr, self.x, self.m, self.node)
            rows = [v.requires_grad_() for v in rows]
            a, _ = self.evaluate(kind, mono, off, rows, rest)
            g = torch.autograd.grad((a * ws[tg].repeat_interleave(count, 0)).sum(), rows)
            gx[tg] += _sums(g[0], count)
            into = [gx, gm] if kind == "leaf" else [gnode[k] for k in ("cm", "mass", "q", "soft")]
            order = torch.argsort(sr)
            per = torch.bincount(sr, minlength=len(into[0]))
            for total, v in zip(into, g[1:]):
                total += _long_sums(v[order], per)
        x, m = self.x.clone().requires_grad_(), self.m.clone().requires_grad_()
        node = _moments(t, x, m, self.e)
        names = sorted(node)
        through = torch.autograd.grad([node[k] for k in names], [x, m], [gnode[k] for k in names])
        ox, om = torch.empty_like(gx), torch.empty_like(gm)
        ox[t.perm], om[t.perm] = gx + through[0], gm + through[1]
        return ox, om


def _sums(v, count, how="sum", initial=0.0):
    return torch.segment_reduce(v, how, lengths=count, axis=0, unsafe=True, initial=initial)


def _long_sums(v, count, how="sum", initial=0.0):
    """_sums in two steps, over parts of at most 256 rows and over the parts
    (one thread sums a segment)."""
    parts = (count + 255) // 256
    owner = torch.arange(len(count), device=count.device).repeat_interleave(parts)
    length = torch.full_like(owner, 256)
    last = torch.cumsum(parts, 0)[count > 0] - 1
    length[last] = (count - 256 * (parts - 1))[count > 0]
    return _sums(_sums(v, length, how, initial), parts, how, initial)


def _ewald(x, root, replicas, side=1.0):
    """LeafEwaldFn: the rest of the lattice of the root's monopole and
    quadrupole, alpha = 2 / L, real-space terms within 2.6 L, 0 < |h| <= 2.8."""
    al = 2.0 / side
    ka = 2.0 * al / math.sqrt(math.pi)
    mass, q = root["mass"], root["q"]
    full = torch.stack([q[0], q[1], q[2], q[1], q[3], q[4], q[2], q[4], q[5]]).reshape(3, 3)
    tr = 0.5 * (q[0] + q[3] + q[5])
    d = x - root["cm"]
    acc = torch.zeros_like(x)
    pot = torch.zeros_like(x[:, 0]) + mass * math.pi / (al * al * side ** 3)
    for rep in itertools.product(range(-3, 4), repeat=3):
        hole = all(abs(k) <= replicas for k in rep)
        r = d + side * torch.tensor(rep, dtype=x.dtype, device=x.device)
        r2 = (r * r).sum(1)
        s2 = r2 * al * al
        series = [ka * (2 * al * al) ** k * (s2 / (2 * k + 3) - 1.0 / (2 * k + 1)) for k in range(4)]
        a = torch.exp(-s2) * ka / r2
        g = [(-torch.erf(al * r2.sqrt()) if hole else torch.erfc(al * r2.sqrt())) * r2.rsqrt()]
        g.append(g[0] / r2 + a)
        g.append(3 * g[1] / r2 + 2 * al ** 2 * a)
        g.append(5 * g[2] / r2 + 4 * al ** 4 * a)
        used = torch.ones_like(r2) if hole else (r2 <= (2.6 * side) ** 2).to(r2)
        g = [used * torch.where(r2 < 1.2e-3 * side * side, s, c) for s, c in zip(series, g)]
        qr = (full[None] * r[:, None, :]).sum(2)
        half = 0.5 * (qr * r).sum(1)
        pot -= g[0] * mass - g[1] * tr + g[2] * half
        acc += g[2][:, None] * qr - r * (g[1] * mass - g[2] * tr + g[3] * half)[:, None]
    w = 2.0 * math.pi / side
    for h in itertools.product(range(-3, 4), repeat=3):
        h2 = sum(k * k for k in h)
        if not 0 < h2 <= 2.8 ** 2:
            continue
        hv = torch.tensor(h, dtype=x.dtype, device=x.device)
        g0 = math.exp(-math.pi ** 2 / (al * al * side * side) * h2) / (math.pi * h2 * side)
        cf = -(g0 * mass - w * w * g0 * 0.5 * (hv[:, None] * full * hv[None]).sum())
        ph = (d * (w * hv)).sum(1)
        pot += cf * torch.cos(ph)
        acc += (cf * torch.sin(ph))[:, None] * (w * hv)
    return acc, pot


def exact(case, seed):
    """run()'s values from the tree algorithm in plain FP64 torch: the same
    interactions, every sum and moment computed directly."""
    case = {**_DEFAULTS, **case}
    if case["n"] > 3000000:
        return None
    pos, vel, mass, soft = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("step", "force", "lists"):
        acc, pot, counters = _Field(case, pos, mass, soft).force()
        return {"values": [*acc.t(), pot], "counters": counters}
    if kind == "vjp":
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        w = torch.randn(case["n"], 3, generator=g, device="cuda", dtype=torch.float64)
        return {"values": list(_Field(case, pos, mass, soft).vjp(w))}
    fields, counters, x, v = [], [0, 0, 0, 0], pos.clone(), vel.clone()
    for _ in range(case["steps"]):
        fields.append(_Field(case, x, mass, soft))
        acc, _, cnt = fields[-1].force()
        counters = [a + b for a, b in zip(counters, cnt)]
        v = v + acc * _DT
        x = x + v * _DT
    if kind == "run":
        return {"values": [*x.t(), *v.t()], "counters": counters}
    lx, lv = 2 * mass[:, None] * x, 2 * mass[:, None] * v
    gm = (v * v).sum(1) + (x * x).sum(1)
    for f in reversed(fields):
        lv = lv + _DT * lx
        gx, g = f.vjp(_DT * lv)
        lx, gm = lx + gx, gm + g
    return {"values": [x, v, lx, lv, gm]}
