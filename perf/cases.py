"""Performance cases: the tree-gravity work that a program has this framework do, through the
calls of gizmo_shared_memory_amd.tree.

A case names one call or one short run of calls (``kind``), the particle distribution it meets and
its sizes. The distributions are those of the package's workloads (Plummer, Hernquist, Hernquist
halo + exponential disk), drawn on the GPU with torch from the seed; previous accelerations (the
relative opening criterion's ``aold``), first radii and velocities come from each profile's closed
form, so that the inputs need no walk of their own.

    build       Morton keys, sort, octree and moments, and the particles in tree order
    walk64      accel_grouped, FP64, the reference's grouping, every particle active
    walk32      accel_grouped, FP32 with the shipped learned criterion, every particle active; its
                result is single precision and is handed on as float32, as an FP32 integrator
                keeps it
    substep     a hierarchical step's small active set on a reused tree: sources re-read, nodes
                refreshed, targets ordered, aold, FP32 walk, accelerations written back
    force       one whole force evaluation with a rebuild (build, order, aold, FP32 walk, write
                back)
    tidal       accel_grouped_tidal with the jerk, every particle active
    potential   the per-target potential walk, every particle
    accel       the per-target acceleration walk on scattered targets (sinks, probes)
    ngb         neighbour lists of about 32 entries around particles
    density     the smoothing-length / density solve, every particle gas

``exact`` is the direct sum over all particles in float64, where it is affordable: a tree walk
approximates it to its opening criterion (about 1e-3).
"""
from __future__ import annotations

import math

import torch

from gizmo_shared_memory_amd import learned
from gizmo_shared_memory_amd import tree as gz

ERR_TOL = 0.0025  # ErrTolForceAcc, the reference's default
GROUP = 64        # targets per group of the FP32 walks: what the autotuner picks from 1M up
EPS = {"plummer": 0.01, "hernquist": 0.005, "halo_disk": 0.005}
PAIRS_MAX = 7.0e10  # direct sums beyond this take too long
F_HALO, RD, ZD = 0.7, 0.1, 0.01  # halo + disk: halo mass share, disk scale length and height

KINDS = ("build", "walk64", "walk32", "substep", "force", "tidal", "potential", "accel", "ngb",
         "density")


def listed():
    return [
        # a star cluster: the smallest tree that is rebuilt every step; launches and read-backs
        dict(name="build_plummer_64k", kind="build", profile="plummer", n=65536, active=65536),
        # a galaxy's tree rebuild: bandwidth of the sort and the level passes
        dict(name="build_hernquist_4m", kind="build", profile="hernquist", n=4194304,
             active=4194304),
        # the parity walk on the small cluster: too few groups to fill the GPU for long
        dict(name="walk64_plummer_64k", kind="walk64", profile="plummer", n=65536, active=65536),
        # the parity walk at galaxy size, the reference's own method in full precision
        dict(name="walk64_hernquist_4m", kind="walk64", profile="hernquist", n=4194304,
             active=4194304),
        # the headline workload: 8M halo + disk, learned criterion, all active
        dict(name="walk32_halo_disk_8m", kind="walk32", profile="halo_disk", n=8388608,
             active=8388608),
        # most force evaluations of a run with hierarchical timesteps: few active, tree reused
        dict(name="substep_halo_disk_1m", kind="substep", profile="halo_disk", n=1048576,
             active=4099),
        # a whole force evaluation of a mid-size run with an odd particle count, tree rebuilt
        dict(name="force_hernquist_262k", kind="force", profile="hernquist", n=262147,
             active=262147),
        # tidal timesteps and jerk: the Hermite-like accuracy options of the walk
        dict(name="tidal_hernquist_1m", kind="tidal", profile="hernquist", n=1048573,
             active=1048573),
        # energy diagnostics
        dict(name="potential_hernquist_1m", kind="potential", profile="hernquist", n=1048576,
             active=1048576),
        # sinks and probes scattered over the domain: the smallest call
        dict(name="accel_hernquist_1m_x1k", kind="accel", profile="hernquist", n=1048576,
             active=1001),
        # hydro's neighbour lists
        dict(name="ngb_hernquist_1m", kind="ngb", profile="hernquist", n=1048576, active=1048576),
        # hydro's smoothing lengths, the costliest single call
        dict(name="density_hernquist_4m", kind="density", profile="hernquist", n=4194304,
             active=4194304, moved=0.01),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    profile = rng.choice(("plummer", "hernquist", "halo_disk"))
    hi = {"build": 4194304, "walk64": 4194304, "walk32": 8388608, "substep": 4194304,
          "force": 2097152, "tidal": 1048576, "potential": 1048576, "accel": 4194304,
          "ngb": 1048576, "density": 4194304}[kind]
    n = _logint(rng, 4000, hi)
    active = n
    if kind == "substep":
        active = _logint(rng, 16, max(17, min(n // 4, 65536)))
    elif kind == "accel":
        active = _logint(rng, 1, min(n, 16384))
    elif kind == "ngb":
        active = _logint(rng, 64, n)
    case = dict(kind=kind, profile=profile, n=n, active=active)
    if kind == "density":  # scatter of the first guesses, in dex
        case["moved"] = round(math.exp(rng.uniform(math.log(0.003), math.log(0.03))), 4)
    return case


# ---- inputs ----------------------------------------------------------------------------------------
def _uniform(g, n):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _isotropic(g, r):
    ct = 2.0 * _uniform(g, r.shape[0]) - 1.0
    st = torch.sqrt(1.0 - ct * ct)
    ph = 2.0 * math.pi * _uniform(g, r.shape[0])
    return r * st * torch.cos(ph), r * st * torch.sin(ph), r * ct


def _hernquist(g, n):
    s = torch.sqrt(_uniform(g, n)) * (50.0 / 51.0)  # truncated at 50 a
    return _isotropic(g, s / (1.0 - s))


def _plummer(g, n):
    u = _uniform(g, n).clamp_(min=1e-12) * (20.0 ** 3 / 401.0 ** 1.5)  # truncated at 20 a
    return _isotropic(g, 1.0 / torch.sqrt(u ** (-2.0 / 3.0) - 1.0))


def _disk(g, n):
    u = _uniform(g, n) * (1.0 - 31.0 * math.exp(-30.0))
    q = torch.full_like(u, 1.7)  # R / Rd, by Newton's method on 1 - (1 + q) exp(-q) = u
    for _ in range(60):
        e = torch.exp(-q)
        q = (q - (1.0 - (1.0 + q) * e - u) / (q * e)).clamp_(1e-12, 30.0)
    ph = 2.0 * math.pi * _uniform(g, n)
    z = -ZD * torch.log(_uniform(g, n).clamp_(min=1e-300))
    z = torch.where(_uniform(g, n) < 0.5, -z, z)
    return RD * q * torch.cos(ph), RD * q * torch.sin(ph), z


def _enclosed(profile, r):
    """Mass inside r (the halo + disk taken as spherical)."""
    hern = (r / (1.0 + r)) ** 2 * (51.0 / 50.0) ** 2
    if profile == "plummer":
        return r ** 3 / (r * r + 1.0) ** 1.5 * (401.0 ** 1.5 / 20.0 ** 3)
    if profile == "hernquist":
        return hern
    return F_HALO * hern + (1.0 - F_HALO) * (1.0 - (1.0 + r / RD) * torch.exp(-r / RD))


def _inputs(case, seed):
    """Positions, masses, softenings, radii, and the state of the generator after them."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + case["n"])
    n, profile = case["n"], case["profile"]
    if profile == "plummer":
        x, y, z = _plummer(g, n)
    elif profile == "hernquist":
        x, y, z = _hernquist(g, n)
    else:
        nh = int(round(F_HALO * n))
        halo, disk = _hernquist(g, nh), _disk(g, n - nh)
        at = torch.randperm(n, generator=g, device="cuda")
        x, y, z = (torch.cat(c)[at] for c in zip(halo, disk))
    m = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    soft = torch.full((n,), EPS[profile], dtype=torch.float64, device="cuda")
    r = torch.sqrt(x * x + y * y + z * z).clamp_(min=1e-9)
    return g, x, y, z, m, soft, r


def _velocities(g, case, r):
    s = torch.sqrt(_enclosed(case["profile"], r) / r / 3.0)
    return tuple(s * torch.randn(case["n"], generator=g, device="cuda", dtype=torch.float64)
                 for _ in range(3))


def _active(g, case, r):
    """Particle indices of the case's active set (int64, ascending)."""
    n, k = case["n"], case["active"]
    if k == n:
        return torch.arange(n, device="cuda")
    if case["kind"] == "substep":  # the shortest timesteps: a noisy dynamical time
        key = 1.5 * torch.log10(r) + 0.5 * torch.randn(n, generator=g, device="cuda",
                                                       dtype=torch.float64)
    else:
        key = _uniform(g, n)
    return torch.sort(torch.topk(key, k, largest=False).indices).values


def _drifted(g, case, x, y, z, r):
    """Substeps: velocities, the time since the build, and the positions then."""
    v = _velocities(g, case, r)
    tau = 1e-4
    return v, tau, tuple((a + tau * b).contiguous() for a, b in zip((x, y, z), v))


def _radius(x, y, z):
    """Radius of about 32 neighbours, for particles in tree order: from the densest run of 17
    consecutive particles that holds each one."""
    k = 17
    if x.shape[0] <= k:
        return torch.full_like(x, float(max(c.max() - c.min() for c in (x, y, z))))
    vol = torch.ones(x.shape[0] - k + 1, dtype=torch.float64, device="cuda")
    for c in (x, y, z):
        run = c.unfold(0, k, 1)
        vol *= run.amax(1) - run.amin(1)
    each = torch.nn.functional.pad((k / vol)[None], (k - 1, k - 1), value=0.0)
    rho = torch.nn.functional.max_pool1d(each, k, stride=1)[0]
    return (32.0 * 3.0 / (4.0 * math.pi * rho)) ** (1.0 / 3.0)


def prepare(case, seed):
    g, x, y, z, m, soft, r = _inputs(case, seed)
    kind, n = case["kind"], case["n"]
    P = gz.Particles(x, y, z, m, soft)
    s = dict(kind=kind, P=P)
    acc = _enclosed(case["profile"], r) / (r * r)  # |a| of the profile, G = 1
    if kind == "build":
        return s
    if kind in ("force", "substep"):
        s["a_prev"] = torch.stack([-acc / r * c for c in (x, y, z)], dim=1).contiguous()
        s["a_grav"] = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    if kind == "force":
        return s
    if kind == "substep":
        v, tau, new = _drifted(g, case, x, y, z, r)
        s["T"] = gz.build(P, vel=v)
        s["active"] = _active(g, case, r).to(torch.int32).view(torch.uint32)
        s["now"], s["tau"] = gz.Particles(*new, m, soft), tau
        return s
    vel = _velocities(g, case, r) if kind == "tidal" else None
    s["T"] = T = gz.build(P, vel=vel)
    s["vel"] = vel
    if kind == "accel":  # in the order of the caller's list, not of the tree
        at = _active(g, case, r)
        at = at[torch.randperm(at.shape[0], generator=g, device="cuda")]
        s["targets"] = at.to(torch.int32).view(torch.uint32)
    elif kind == "ngb":
        at = torch.zeros(n, dtype=torch.bool, device="cuda")
        at[_active(g, case, r)] = True
        order = T.device_orderbuf().view(torch.int32).long()
        at = order[at[order]]  # the queries in tree order
        s["centres"] = torch.stack([c[at] for c in (x, y, z)], dim=1).contiguous()
        h = torch.empty_like(x)
        h[order] = _radius(x[order], y[order], z[order])
        s["radius"] = h[at]
        s["lists"] = torch.zeros(128 * at.shape[0], dtype=torch.int32, device="cuda")
        return s
    else:
        s["targets"] = T.device_orderbuf()
    at = s["targets"].view(torch.int32).long()
    if kind == "density":  # first guesses: the radii of the step before, from which these moved
        h = gz.density(T, P, s["targets"], 32.0, 1.0, h_start=_radius(x[at], y[at], z[at]))[0]
        s["h"] = h * 10.0 ** (case["moved"] * torch.randn(n, generator=g, device="cuda",
                                                          dtype=torch.float64))
        return s
    s["aold"] = (ERR_TOL * acc)[at]
    if kind == "walk32":
        s["model"] = learned.load_model()
    return s


def run(s):
    kind, P = s["kind"], s["P"]
    if kind == "build":
        T = gz.build(P)
        return {"order": T.device_orderbuf().view(torch.int32), "nnodes": T.nnodes}
    if kind == "force":
        T = gz.build(P)
        tg = gz.order_targets(T)
        aold = gz.aold_from_accel(T, s["a_prev"], tg, ERR_TOL)
        a = gz.accel_grouped(T, P, tg, 0.0, aold=aold, precision="fp32", group_size=GROUP)
        gz.scatter_accel(tg, *a, s["a_grav"])
        return s["a_grav"]
    T = s["T"]
    if kind == "substep":
        now = s["now"]
        T.update_sources(now)
        T.refresh_walk_nodes(s["tau"])
        tg = gz.order_targets(T, s["active"])
        aold = gz.aold_from_accel(T, s["a_prev"], tg, ERR_TOL)
        a = gz.accel_grouped(T, now, tg, 0.0, aold=aold, precision="fp32", group_size=GROUP)
        gz.scatter_accel(tg, *a, s["a_grav"])
        return s["a_grav"]
    if kind == "ngb":
        start, found = gz.ngb_search(T, s["centres"], s["radius"])
        s["lists"][:found.shape[0]] = found.view(torch.int32)  # the program's own buffer
        return {"start": start, "lists": s["lists"]}
    tg = s["targets"]
    if kind == "density":
        h, rho, nngb, iters = gz.density(T, P, tg, 32.0, 1.0, h_start=s["h"])
        return {"h": h, "rho": rho, "nngb": nngb, "iters": iters}
    aold = s["aold"]
    if kind == "walk64":
        return gz.accel_grouped(T, P, tg, 0.0, aold=aold)
    if kind == "walk32":
        a = gz.accel_grouped(T, P, tg, 0.0, aold=aold, precision="fp32", group_size=GROUP,
                             model=s["model"])
        return tuple(c.float() for c in a)
    if kind == "tidal":
        ax, ay, az, tid, jerk = gz.accel_grouped_tidal(T, P, tg, 0.0, aold=aold, vel=s["vel"],
                                                       jerk=True)
        return {"a": (ax, ay, az), "tidal": tid, "jerk": jerk}
    if kind == "potential":
        return gz.potential(T, P, tg, 0.0, aold=aold)
    return gz.accel(T, P, tg, 0.0, aold=aold)


# ---- the direct sum ----------------------------------------------------------------------------------
def _inside(u, h):
    """Force over r, potential and tidal factor of the cubic-spline kernel of extent h, u = r/h < 1."""
    u = u.clamp(min=1e-30)
    lo = u < 0.5
    force = torch.where(lo, 32.0 / 3.0 + u * u * (32.0 * u - 38.4),
                        64.0 / 3.0 - 48.0 * u + 38.4 * u * u - 32.0 / 3.0 * u ** 3
                        - 1.0 / (15.0 * u ** 3)) / h ** 3
    pot = torch.where(lo, -2.8 + u * u * (16.0 / 3.0 + u * u * (6.4 * u - 9.6)),
                      -3.2 + 1.0 / (15.0 * u) + u * u * (32.0 / 3.0 + u * (-16.0 + u * (
                          9.6 - 32.0 / 15.0 * u)))) / h
    tide = torch.where(lo, 76.8 - 96.0 * u,
                       -0.2 / u ** 5 + 48.0 / u - 76.8 + 32.0 * u) / h ** 5
    return force, pot, tide


def _direct(want, x, y, z, m, h, targets, vel=None):
    """Direct sums of the targets with a common kernel extent h: rows (ax, ay, az) for "a", phi
    for "phi", and for "tidal" the acceleration, tidal tensor (xx yy zz xy yz xz) and jerk."""
    n = x.shape[0]
    out = torch.empty({"a": 3, "phi": 1, "tidal": 12}[want], targets.shape[0],
                      dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // n)
    for lo in range(0, targets.shape[0], step):
        at = targets[lo:lo + step]
        d = [c[None, :] - c[at][:, None] for c in (x, y, z)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        near = torch.nonzero(r2 < h * h, as_tuple=True)  # the targets themselves among them
        rn = torch.sqrt(r2[near])
        force, pot, tide = _inside(rn / h, h)
        itself = rn == 0.0
        r2[near] = 1.0
        inv = torch.rsqrt(r2)
        rows = out[:, lo:lo + step]
        if want == "phi":
            inv.neg_()
            inv[near] = torch.where(itself, 0.0, pot)
            rows[0] = inv @ m
            continue
        f = inv * inv * inv
        if want == "tidal":
            t = 3.0 * f * inv * inv
            t[near] = torch.where(itself, 0.0, tide)
            t *= m
        f[near] = torch.where(itself, 0.0, force)
        f *= m
        for k in range(3):
            rows[k] = (f * d[k]).sum(1)
        if want == "tidal":
            trace = f.sum(1)
            for k, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))):
                rows[3 + k] = (t * d[i] * d[j]).sum(1) - (trace if i == j else 0.0)
            dv = [c[None, :] - c[at][:, None] for c in vel]
            t *= dv[0] * d[0] + dv[1] * d[1] + dv[2] * d[2]
            for k in range(3):
                rows[9 + k] = (f * dv[k] - t * d[k]).sum(1)
    return out


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    # the other calls return whole numbers, or radii that the solve's tolerance leaves open
    if kind in ("build", "ngb", "density"):
        return None
    if float(n) * case["active"] * (4.0 if kind == "tidal" else 1.0) > PAIRS_MAX:
        return None
    g, x, y, z, m, soft, r = _inputs(case, seed)
    h = EPS[case["profile"]]
    if kind == "substep":
        _, _, (x, y, z) = _drifted(g, case, x, y, z, r)
        at = _active(g, case, r)
        out = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
        out[at] = _direct("a", x, y, z, m, h, at).t()
        return out
    if kind == "force":
        return _direct("a", x, y, z, m, h, torch.arange(n, device="cuda")).t().contiguous()
    vel = _velocities(g, case, r) if kind == "tidal" else None
    if kind == "accel":
        at = _active(g, case, r)
        at = at[torch.randperm(at.shape[0], generator=g, device="cuda")]
    else:
        at = _order(x, y, z)
    if kind == "potential":
        return _direct("phi", x, y, z, m, h, at)[0]
    if kind == "tidal":
        rows = _direct("tidal", x, y, z, m, h, at, vel)
        return {"a": tuple(rows[:3]), "tidal": rows[3:9], "jerk": rows[9:12]}
    return tuple(_direct("a", x, y, z, m, h, at))


def _order(x, y, z):
    """Particles in Morton order: 20 bits an axis of the cube about the bounding box's centre whose
    side is 1.0000001 of its largest, z the highest bit, ties in the order of the particles."""
    lo = [float(c.min()) for c in (x, y, z)]
    hi = [float(c.max()) for c in (x, y, z)]
    side = max(b - a for a, b in zip(lo, hi)) * 1.0000001
    scale = float((1 << 20) - 1) / side
    key = torch.zeros(x.shape[0], dtype=torch.int64, device="cuda")
    for axis, c in enumerate((x, y, z)):
        q = ((c - (0.5 * (lo[axis] + hi[axis]) - 0.5 * side)) * scale).to(torch.int64)
        for b in range(20):
            key |= ((q >> b) & 1) << (3 * b + axis)
    return torch.sort(key, stable=True).indices


# ---- the work that a pass cannot do without -------------------------------------------------------------
def work(case):
    n, k, kind = float(case["n"]), float(case["active"]), case["kind"]
    # interactions per target at ErrTolForceAcc = 0.0025 (1,154 counted at 8M halo + disk)
    inter = 50.0 * math.log2(n)
    build_bytes = 40.0 * n + 75.0 * n  # particles in; order, ranks, leaves, sorted copy, nodes out
    walk_bytes = 55.0 * n + 56.0 * k   # sources and nodes; target, aold and result
    if kind == "build":
        return {"bytes": build_bytes + 4.0 * n, "flops": 20.0 * n}
    if kind == "force":
        return {"bytes": build_bytes + walk_bytes + 72.0 * k, "flops": 20.0 * inter * k}
    if kind == "substep":
        return {"bytes": 40.0 * n + walk_bytes + 72.0 * k, "flops": 20.0 * inter * k}
    if kind == "tidal":
        return {"bytes": walk_bytes + 24.0 * n + 96.0 * k, "flops": 66.0 * inter * k}
    if kind == "accel":  # scattered targets reach a small part of a large tree
        return {"bytes": min(55.0 * n, 40.0 * inter * k) + 56.0 * k, "flops": 20.0 * inter * k}
    if kind == "ngb":    # centre and radius in, 32 entries out; about four candidates an entry
        return {"bytes": 40.0 * n + (32.0 + 8.0 + 128.0) * k, "flops": 8.0 * 128.0 * k}
    if kind == "density":  # 32 neighbours in each of about three iterations
        return {"bytes": 48.0 * n + 32.0 * k, "flops": 40.0 * 32.0 * 3.0 * k}
    return {"bytes": walk_bytes, "flops": 20.0 * inter * k}
