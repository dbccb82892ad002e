"""The work this library is measured on: which cases, their inputs, one pass, and what a pass computes in 64 bits.

Every case goes through the public entry points of grasph2_amd (the C ABI of include/grasph2.h) on
device-resident particles, as a simulation's main loop does: derivatives, then the leapfrog.  Time steps
are short, so that thousands of passes leave a state the kind of state its case stands for.

Kinds:
  nbody      self-gravity alone: a Plummer sphere, equal or unequal masses
  default    the settings a user starts from (grasph_params_default): solids with integrated density,
             Mohr-Coulomb plasticity and the variable-step leapfrog, one sphere
  liquid     a liquid blob with self-gravity, with or without XSPH
  collision  two solid spheres just out of reach, or overlapping (in contact)
  impact     a solid body squeezed by an impact: hundreds of neighbours per particle in its core
  passes     the three pair passes called one by one on bodies in contact
  nogravity  two solid spheres in contact without self-gravity (laboratory impacts)
  noalloc    the allocation-free entry point on a collision
  ensemble   many independent collisions advanced together by grasph_batch_step
  large      one rotating solid sphere with unequal masses
"""
import math

import numpy as np
import torch

import grasph2_amd as g
from grasph2_amd import ics

DEV = "cuda"
DT = 1e-5


def listed():
    return [
        # the smallest calls: a star cluster of a thousand bodies, where launches and latency count
        {"name": "nbody_1000", "kind": "nbody", "n": 1000, "equal": True},
        # the N-body benchmark configuration
        {"name": "nbody_16384", "kind": "nbody", "n": 16384, "equal": True},
        # a ragged count with a mass spectrum
        {"name": "nbody_50021_masses", "kind": "nbody", "n": 50021, "equal": False},
        # what a user gets who changes no setting
        {"name": "default_16384", "kind": "default", "n": 16384},
        # the liquid benchmark configuration
        {"name": "liquid_65536", "kind": "liquid", "n": 65536, "xsph": False},
        # the headline configuration
        {"name": "collision_131072", "kind": "collision", "n": 131072, "gap": 1.0},
        # the same simulation once the bodies have hit: long neighbour lists
        {"name": "impact_65536", "kind": "impact", "n": 65536, "squeeze": 0.55},
        # a caller that runs the passes itself
        {"name": "passes_20011", "kind": "passes", "n": 20011, "gap": -2.0},
        # SPH alone: neighbour search and passes, no all-pairs gravity
        {"name": "nogravity_200003", "kind": "nogravity", "n": 200003, "gap": -2.0},
        # serving loops that may not allocate
        {"name": "noalloc_8192", "kind": "noalloc", "n": 8192, "gap": 1.0},
        # the batched-ensemble benchmark configuration
        {"name": "ensemble_512", "kind": "ensemble", "count": 512, "nmin": 1024, "nmax": 16384},
        # the largest configuration
        {"name": "large_1048576", "kind": "large", "n": 1048576},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["nbody", "nbody", "default", "liquid", "collision", "collision", "impact", "passes",
                       "nogravity", "noalloc", "ensemble", "large"])
    if kind == "nbody":
        return {"kind": kind, "n": _log_size(rng, 700, 131072), "equal": rng.random() < 0.5}
    if kind == "default":
        return {"kind": kind, "n": _log_size(rng, 2048, 131072)}
    if kind == "liquid":
        return {"kind": kind, "n": _log_size(rng, 2048, 131072), "xsph": rng.random() < 0.5}
    if kind == "collision":
        return {"kind": kind, "n": _log_size(rng, 2048, 262144), "gap": rng.choice([1.0, -2.0])}
    if kind == "impact":
        return {"kind": kind, "n": _log_size(rng, 16384, 131072), "squeeze": round(rng.uniform(0.5, 0.7), 3)}
    if kind == "passes":
        return {"kind": kind, "n": _log_size(rng, 2048, 65536), "gap": rng.choice([1.0, -2.0])}
    if kind == "nogravity":
        return {"kind": kind, "n": _log_size(rng, 8192, 400000), "gap": rng.choice([1.0, -2.0])}
    if kind == "noalloc":
        return {"kind": kind, "n": _log_size(rng, 1024, 40000), "gap": rng.choice([1.0, -2.0])}
    if kind == "ensemble":
        nmin = rng.choice([512, 1024, 2048])
        return {"kind": kind, "count": _log_size(rng, 8, 512), "nmin": nmin, "nmax": rng.choice([4096, 8192, 16384])}
    return {"kind": kind, "n": _log_size(rng, 262144, 1048576)}


# ---------------------------------------------------------------- inputs

def _lattice_sites(n):
    """The n sites of the integer cubic lattice closest to the origin, closest first."""
    m = int(math.ceil((3.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0))) + 2
    a = torch.arange(-m, m + 1, device=DEV)
    s = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), dim=-1).reshape(-1, 3)
    order = torch.sort((s * s).sum(1), stable=True).indices[:n]
    return s[order].double()


def _spacing(n):
    """Lattice spacing of n sites in the unit sphere."""
    return (4.0 / 3.0 * math.pi / n) ** (1.0 / 3.0)


def _rand(gen, *shape):
    return torch.rand(shape, generator=gen, device=DEV, dtype=torch.float64)


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float64)


def _sizes(case):
    """Particle counts of an ensemble's instances: the case's, whatever the seed."""
    return np.random.default_rng(4).integers(case["nmin"], case["nmax"] + 1, size=case["count"])


def _plummer(n, gen, equal):
    def iso(k):
        u = 2.0 * _rand(gen, k) - 1.0
        phi = 2.0 * math.pi * _rand(gen, k)
        s = torch.sqrt(1.0 - u * u)
        return torch.stack([s * torch.cos(phi), s * torch.sin(phi), u], 1)

    cut = (10.0 ** -2 + 1.0) ** -1.5  # mass inside r = 10
    r = 1.0 / torch.sqrt((cut * _rand(gen, n)).clamp_min(1e-12) ** (-2.0 / 3.0) - 1.0)
    pos = iso(n) * r[:, None]
    # speeds as fractions of the escape speed with density q^2 (1 - q^2)^3.5
    q = (_rand(gen, 16 * n), 0.1 * _rand(gen, 16 * n))
    q = q[0][q[1] < q[0] ** 2 * (1.0 - q[0] ** 2) ** 3.5]
    q = q[torch.arange(n, device=DEV) % q.numel()]
    vel = iso(n) * (q * math.sqrt(2.0) * (1.0 + r * r) ** -0.25)[:, None]
    mass = torch.ones(n, device=DEV, dtype=torch.float64) if equal else _rand(gen, n).clamp_min(1e-3) ** -0.7
    mass = mass / mass.sum()
    pos = pos - (pos * mass[:, None]).sum(0)
    vel = vel - (vel * mass[:, None]).sum(0)
    return pos, vel, mass


def _spheres(n, gen, gap, speed, angle_deg, sites):
    """Two jittered lattice spheres of unit radius; gap: their separation in units of H."""
    na = n // 2
    nb = n - na
    d = _spacing(na)
    H = 2.5 * d
    sep = 2.0 + gap * H

    def ball(k):
        dk = _spacing(k)
        return sites[:k] * dk + (2.0 * _rand(gen, k, 3) - 1.0) * (0.1 * dk)

    shift = torch.tensor([sep / 2, 0.0, 0.0], device=DEV, dtype=torch.float64)
    pos = torch.cat([ball(na) - shift, ball(nb) + shift])
    th = math.radians(angle_deg)
    u = torch.tensor([math.cos(th), math.sin(th), 0.0], device=DEV, dtype=torch.float64)
    vel = torch.cat([(u * speed * nb / n).expand(na, 3), (-u * speed * na / n).expand(nb, 3)])
    return pos, vel + 0.02 * _normal(gen, n, 3), d, H


def _planes(v, k):
    return v.t().contiguous().reshape(k, -1)


def _fields(pos, vel, mass, rho, solid, gen, stress=0.01):
    """The particle arrays of include/grasph2.h."""
    n = pos.shape[0]
    f32 = dict(device=DEV, dtype=torch.float32)
    posm = torch.empty((n, 4), **f32)
    posm[:, :3] = pos
    posm[:, 3] = mass
    v4 = torch.zeros((n, 4), **f32)
    v4[:, :3] = vel
    a = {"posm": posm, "pos64": _planes(posm[:, :3].double(), 3), "vel": v4, "acc": torch.zeros((n, 4), **f32)}
    if rho is not None:
        a["density"] = torch.full((n,), rho, **f32)
        a["maxvsig"] = torch.zeros(n, **f32)
        if solid:
            a["balsara"] = torch.zeros(n, **f32)
            a["density_dt"] = torch.zeros(n, **f32)
            s = stress * _normal(gen, 6, n)
            s[2] = -s[0] - s[1]
            a["dstress"] = s.float()
            a["dstress_dt"] = torch.zeros((6, n), **f32)
        else:
            a["xvel"] = torch.zeros((n, 4), **f32)
    return a


def _instances(case, seed):
    """[(particle arrays, parameters)] of a case: one, or an ensemble's."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 1000003 + 17)
    kind = case["kind"]
    if kind == "nbody":
        pos, vel, mass = _plummer(case["n"], gen, case["equal"])
        return [(_fields(pos, vel, mass, None, False, gen), ics.plummer_params(0.01, DT))]
    if kind == "ensemble":
        rng = np.random.default_rng(seed)
        sizes = _sizes(case)
        sites = _lattice_sites((case["nmax"] + 1) // 2 + 1)
        out = []
        for n in sizes:
            pos, vel, d, H = _spheres(int(n), gen, 1.0, rng.uniform(0.1, 1.0), rng.uniform(0.0, 60.0), sites)
            out.append((_fields(pos, vel, d ** 3, 1.0, True, gen), ics.solid_params(H, DT)))
        return out
    n = case["n"]
    if kind == "default":
        prm = g.default_params()
        # the default body: unit mass in a sphere of radius 0.1, H and the rest density scaled to the count
        scale = (16384.0 / n) ** (1.0 / 3.0)
        prm.H *= scale
        prm.normalsep *= scale
        prm.initial_timestep, prm.min_timestep, prm.max_timestep = 1e-6, 1e-7, 1e-6
        pos = _lattice_sites(n) * (0.1 * _spacing(n))
        pos = pos + (2.0 * _rand(gen, n, 3) - 1.0) * (0.01 * _spacing(n))
        return [(_fields(pos, 0.05 * _normal(gen, n, 3), 1.0 / n, prm.rho0, True, gen, 0.1), prm)]
    if kind == "liquid":
        d = _spacing(n)
        pos = _lattice_sites(n) * d + (2.0 * _rand(gen, n, 3) - 1.0) * (0.1 * d)
        prm = ics.liquid_params(2.5 * d, DT)
        if case["xsph"]:
            prm.flags |= g.XSPH
        return [(_fields(pos, 0.05 * _normal(gen, n, 3), d ** 3, 1.0, False, gen), prm)]
    if kind == "large":
        d = _spacing(n)
        pos = _lattice_sites(n) * d
        mass = d ** 3 * (0.99 + 0.02 * _rand(gen, n))
        om = 0.3 * math.sqrt(float(mass.sum()))
        vel = torch.stack([-om * pos[:, 1], om * pos[:, 0], torch.zeros_like(pos[:, 0])], 1)
        return [(_fields(pos, vel, mass, 1.0, True, gen), ics.solid_params(2.5 * d, DT))]
    if kind == "impact":
        d = _spacing(n)
        pos = _lattice_sites(n) * d + (2.0 * _rand(gen, n, 3) - 1.0) * (0.1 * d)
        r = pos.norm(dim=1, keepdim=True).clamp_min(1e-9)
        pos = pos * (case["squeeze"] * r ** 0.3)  # compressed, most towards the centre
        prm = ics.solid_params(2.5 * d, DT)
        return [(_fields(pos, -0.2 * pos + 0.05 * _normal(gen, n, 3), d ** 3, 1.0, True, gen), prm)]
    pos, vel, d, H = _spheres(n, gen, case["gap"], 0.5, 30.0, _lattice_sites((n + 1) // 2))
    prm = ics.solid_params(H, DT, gravity=kind != "nogravity")
    return [(_fields(pos, vel, d ** 3, 1.0, True, gen), prm)]


def _view(a):
    v = g.Particles()
    v.n = a["posm"].shape[0]
    for f, t in a.items():
        setattr(v, f, t.data_ptr())
    return v


class State:
    """One context and its particles, as a program keeps them."""

    def __init__(self, case, seed):
        self.kind = case["kind"]
        inst = _instances(case, seed)
        self.ctx = g.Context(torch.cuda.current_device())
        if self.kind == "ensemble":
            # the batch layout: every array the concatenation of the instances' own
            self.arrays = {f: torch.cat([a[f].reshape(-1) for a, _ in inst]) for f in inst[0][0]}
            self.arrays = {f: t.reshape(-1, 4) if f in ("posm", "vel", "acc") else t for f, t in self.arrays.items()}
            offsets = np.concatenate([[0], np.cumsum([a["posm"].shape[0] for a, _ in inst])])
            self.batch = self.ctx.batch(offsets, [p for _, p in inst])
        else:
            self.arrays, self.prm = inst[0]
        self.view = _view(self.arrays)


def prepare(case, seed):
    return State(case, seed)


def run(state):
    ctx, view = state.ctx, state.view
    if state.kind == "ensemble":
        ctx.batch_step(view, state.batch, 1)
        return state.arrays
    prm = state.prm
    if state.kind == "passes":
        ctx.calc_density(view, prm)
        ctx.calc_balsara_density_dt_dstress_dt(view, prm)
        ctx.calc_acceleration(view, prm)
        return {f: state.arrays[f] for f in ("density", "balsara", "dstress_dt", "maxvsig", "acc")}
    if state.kind == "noalloc":
        ctx.compute_derivatives_noalloc(view, prm)
    else:
        ctx.compute_derivatives(view, prm)
    ctx.integrate(view, prm, True)
    return state.arrays


# ---------------------------------------------------------------- the work of one pass

def work(case):
    """20 operations per ordered gravity pair; per neighbour pair (about 65 of them within 2.5 spacings) the
    passes' formulas; every particle array read once, and once written where the pass changes it."""
    kind = case["kind"]
    if kind == "ensemble":
        sizes = _sizes(case).astype(float)
    else:
        sizes = np.array([float(case["n"])])
    n, pairs = float(sizes.sum()), float((sizes * (sizes - 1.0)).sum())
    flops = 0.0 if kind == "nogravity" else 20.0 * pairs
    if kind == "nbody":
        return {"bytes": n * (16 + 24 + 16 + 12 + 24 + 16 + 16), "flops": flops}
    near = 4.0 / 3.0 * math.pi * 2.5 ** 3 * n
    if kind == "impact":
        near *= 6.0
    flops += near * (73.0 if kind == "liquid" else 147.5 if kind == "default" else 165.0)
    per = 16 + 24 + 16 + 12 + 24 + 16 + 16 + 8 + 4 + (16 if kind == "liquid" else 4 * (6 + 6 + 6) + 8)
    return {"bytes": n * per, "flops": flops}


# ---------------------------------------------------------------- the same in 64 bits

_TERMS = 1 << 27  # pair values held at once


def _pairs_and_gravity(x, m, H2, grav, sph):
    """Gravity of every particle and the ordered pairs (i, j) with 0 < r^2 <= H^2."""
    n = x.shape[0]
    acc = torch.zeros_like(x)
    ii, jj = [], []
    step = max(1, _TERMS // n)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [x[None, :, c] - x[a:b, None, c] for c in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        if sph:
            near = ((r2 <= H2) & (r2 > 0.0)).nonzero()
            ii.append((near[:, 0] + a).int())
            jj.append(near[:, 1].int())
            del near
        if grav:
            s = (r2 + H2) if H2 > 0.0 else torch.where(r2 > 0.0, r2, torch.full_like(r2, math.inf))
            del r2
            s = s.rsqrt_()
            s = s * s * s * m[None, :]
            for c in range(3):
                acc[a:b, c] = (s * d[c]).sum(1)
            del s
        del d
    if not sph:
        return acc, None, None
    return acc, torch.cat(ii).long(), torch.cat(jj).long()


def _sum(n, i, v):
    return torch.zeros((n,) + v.shape[1:], dtype=v.dtype, device=v.device).index_add_(0, i, v)


def _sym(t6):
    xx, yy, zz, xy, xz, yz = t6
    return torch.stack([torch.stack([xx, xy, xz], -1), torch.stack([xy, yy, yz], -1), torch.stack([xz, yz, zz], -1)], -2)


def _unique(t):
    return torch.stack([t[:, 0, 0], t[:, 1, 1], t[:, 2, 2], t[:, 0, 1], t[:, 0, 2], t[:, 1, 2]])


def _derivatives(a, p):
    """Derivatives of one instance's arrays (float64 dict in and out)."""
    f = p.flags
    n = a["posm"].shape[0]
    x, m, v = a["posm"][:, :3], a["posm"][:, 3], a["vel"][:, :3]
    H = float(p.H)
    sph, grav, solid = bool(f & g.SPH), bool(f & g.SELF_GRAVITY), bool(f & g.SOLIDS)
    acc, i, j = _pairs_and_gravity(x, m, H * H, grav, sph)
    out = {}
    if sph:
        r_ij = x[i] - x[j]
        r = r_ij.norm(dim=1)
        q = r / H
        w = 8.0 / (math.pi * H ** 3) * torch.where(q < 0.5, 6 * q ** 3 - 6 * q ** 2 + 1, 2 * (1 - q).clamp_min(0) ** 3)
        dw = 48.0 / (math.pi * H ** 4) * torch.where(q < 0.5, (3 * q - 2) / H, -((1 - q).clamp_min(0) ** 2) / r)
        grad = dw[:, None] * r_ij
        vij = v[i] - v[j]
        mj = m[j]
        rho = a["density"]
        if not f & g.INTEGRATE_DENSITY:
            rho = _sum(n, i, mj * w)
            out["density"] = rho
        vol = mj / rho[j]
        bal = torch.ones_like(rho)
        S = _sym(a["dstress"]) if solid else None
        if solid or f & (g.INTEGRATE_DENSITY | g.BALSARA_SWITCH):
            vg = vij[:, :, None] * grad[:, None, :]
            G = -_sum(n, i, vol[:, None, None] * vg)  # velocity gradient: e + rotation
            div = G.diagonal(dim1=1, dim2=2).sum(1)
            e, rot = 0.5 * (G + G.transpose(1, 2)), 0.5 * (G - G.transpose(1, 2))
            if solid:
                eye = torch.eye(3, device=DEV, dtype=torch.float64)
                sdt = 2.0 * p.shear * (e - eye * (div / 3.0)[:, None, None])
                sdt = sdt + S @ rot.transpose(1, 2) + rot @ S.transpose(1, 2)
                out["dstress_dt"] = _unique(sdt)
            if f & g.BALSARA_SWITCH:
                curl = 2.0 * torch.stack([rot[:, 1, 2], rot[:, 0, 2], rot[:, 0, 1]], 1).norm(dim=1)
                bal = div.abs() / (div.abs() + curl + 0.0001 * p.SOUNDSPEED / H)
                out["balsara"] = bal
            out["density_dt"] = -rho * div if f & g.INTEGRATE_DENSITY else torch.zeros_like(rho)
            del vg, G
        if solid:
            pres = p.BULK / p.dBULKdP * ((rho / p.rho0) ** p.dBULKdP - 1.0)
            sig = (S - pres[:, None, None] * torch.eye(3, device=DEV, dtype=torch.float64)) / (rho * rho)[:, None, None]
            F = mj[:, None] * ((sig[i] + sig[j]) @ grad[:, :, None])[:, :, 0]
        else:
            sig = -(p.SOUNDSPEED ** 2) * (rho - p.rho0) / (rho * rho)
            F = (mj * (sig[i] + sig[j]))[:, None] * grad
        maxv = torch.zeros(n, device=DEV, dtype=torch.float64)
        if f & g.ARTIFICIAL_VISCOSITY:
            wij = (r_ij * vij).sum(1) / r
            vsig = 2.0 * p.SOUNDSPEED - 3.0 * wij
            visc = -0.25 * (bal[i] + bal[j]) * p.alpha * wij * vsig / (0.5 * (rho[i] + rho[j]))
            visc = torch.where(wij < 0.0, visc, torch.zeros_like(visc))
            F = F - (mj * visc)[:, None] * grad
            if f & g.BALSARA_SWITCH:
                maxv.scatter_reduce_(0, i, torch.where(wij < 0.0, vsig, torch.zeros_like(vsig)), "amax")
        out["maxvsig"] = maxv
        acc = acc + _sum(n, i, F)
        if "xvel" in a:
            xv = torch.zeros((n, 4), device=DEV, dtype=torch.float64)
            if f & g.XSPH:
                xv[:, :3] = _sum(n, i, (2.0 * mj / (rho[i] + rho[j]) * w)[:, None] * (v[j] - v[i]))
            out["xvel"] = xv
    out["acc"] = torch.cat([acc, torch.zeros((n, 1), device=DEV, dtype=torch.float64)], 1)
    return out


def _leapfrog(a, p):
    """integrate(pb, true) on one instance's arrays (float64, derivatives in place)."""
    f = p.flags
    dt, kick = float(p.fixed_timestep), float(p.fixed_timestep)
    if f & g.VARIABLE_TIMESTEP:  # a new context: current dt is 0, next dt max_timestep
        la = a["acc"][:, :3].norm(dim=1)
        dt = min(float(p.max_timestep), float((p.accel_accuracy * p.H / la).sqrt().min()),
                 float((p.velocity_accuracy * p.H / a["maxvsig"]).min()))
        dt = max(dt, float(p.min_timestep))
        kick = 0.5 * dt
    o = dict(a)
    v = a["vel"][:, :3] + a["acc"][:, :3] * kick
    u = v + p.xsph_factor * a["xvel"][:, :3] if f & g.XSPH else v
    o["pos64"] = a["pos64"] + u.t() * dt
    o["posm"] = torch.cat([o["pos64"].t(), a["posm"][:, 3:]], 1)
    o["vel"] = torch.cat([v, a["vel"][:, 3:]], 1)
    if f & g.SPH:
        if f & g.INTEGRATE_DENSITY:
            o["density"] = (a["density"] + a["density_dt"] * dt).clamp_min(0.0)
        if f & g.SOLIDS:
            S = a["dstress"] + a["dstress_dt"] * dt
            J2 = 0.5 * (S[0] ** 2 + S[1] ** 2 + S[2] ** 2) + S[3] ** 2 + S[4] ** 2 + S[5] ** 2
            if f & g.PLASTICITY_MC:
                Y = p.tanfr * (p.BULK / p.dBULKdP * ((o["density"] / p.rho0) ** p.dBULKdP - 1.0)) + p.cohesion
            else:
                Y = torch.full_like(J2, p.Y)
            o["dstress"] = S * torch.where(Y * Y < 3.0 * J2, Y * Y / (3.0 * J2), torch.ones_like(J2))
    return o


def exact(case, seed):
    if case["kind"] == "large":
        return None  # 2.7e11 to 1.1e12 pairs in 64 bits
    outs = []
    for arrays, prm in _instances(case, seed):
        a = {f: t.double() for f, t in arrays.items()}
        a.update(_derivatives(a, prm))
        outs.append(a if case["kind"] == "passes" else _leapfrog(a, prm))
    if case["kind"] == "passes":
        return {f: outs[0][f] for f in ("density", "balsara", "dstress_dt", "maxvsig", "acc")}
    if case["kind"] != "ensemble":
        return outs[0]
    o = {f: torch.cat([a[f].reshape(-1) for a in outs]) for f in outs[0]}
    return {f: t.reshape(-1, 4) if f in ("posm", "vel", "acc") else t for f, t in o.items()}
