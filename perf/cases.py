"""Workloads that the library's performance is followed on, each through the
entry points a program calls: whole unbinding calls from one subhalo to a large
population, the learned snapshot step, a resident batch with its profiles, the
gravity tree, the exact sum, particle reassignment and the classifier.

Sizes come from the benchmark and the tests: the 12,000-particle NFW halo, the
power-law population on [20, 10^6] particles, the hydro mixture, the NFW host
with 50 embedded subhaloes, host haloes with 79% tracers.  Particles are drawn on
the GPU (NFW members in Jeans equilibrium plus fast interlopers, as synth.py
draws them) and handed over as the host arrays the library takes.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hbt-herons_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import hbtx  # noqa: E402
import learned  # noqa: E402
import synth  # noqa: E402

MASS = synth.PARTICLE_MASS
_shared = {}


def context():
    """The program's one context (a program keeps one per host thread)."""
    if "ctx" not in _shared:
        _shared["ctx"] = hbtx.Context(0)
    return _shared["ctx"]


# --- the cases ---------------------------------------------------------------------

def listed():
    return [
        # one small subhalo through the per-subhalo drop-in of Subhalo_t::Unbind: launches and latency
        dict(name="one_subhalo_300", kind="one", n=300, plain=True, bmp=0.995),
        # the benchmark's single NFW halo of 10,000 particles and 2,000 interlopers
        dict(name="one_halo_12k", kind="one", n=12000, plain=False, bmp=0.995),
        # many small subhaloes (20 to 2,000 particles), the bulk of a snapshot's subhaloes by number
        dict(name="small_subhaloes_1.2m", kind="batch", n=1_200_011, nmax=2000, hydro=False, defaults=False, bmp=0.995),
        # the power-law population of the benchmark (about 20,000 subhaloes up to 10^6 particles)
        dict(name="population_8m", kind="batch", n=8_000_000, nmax=1_000_000, hydro=False, defaults=False, bmp=0.995),
        # the hydro mixture with particle types, thermal energy and iteration to the fixed point
        dict(name="hydro_2.1m", kind="batch", n=2_135_724, nmax=1_000_000, hydro=True, defaults=False, bmp=1.0),
        # the reference's default parameters: periodic box, subsampled potentials, centre refinement
        dict(name="defaults_periodic_1m", kind="batch", n=1_000_003, nmax=300_000, hydro=False, defaults=True, bmp=0.995),
        # a snapshot unbound from the previous one's outputs: load, features, inference, warm start, fetch
        dict(name="learned_snapshot_4m", kind="learned", n=4_000_000, nmax=1_000_000, min_particles=30000, bmp=0.995),
        # inputs resident in device memory: iterate, save potentials, profiles and shapes, results to the host
        dict(name="resident_profiles_3m", kind="resident", n=3_000_017, nmax=1_000_000, bmp=1.0),
        # GravityTree_t: one tree over the NFW host with 50 subhaloes, potential at every particle
        dict(name="tree_host_2m", kind="tree", n=2_000_000, nsub=50),
        # exact potentials from device arrays without allocation (a serving loop)
        dict(name="direct_30k_on_20k", kind="direct", n_src=20_011, n_tgt=30_001, periodic=False),
        # reassignment of gas to the nearest tracers' subhaloes, the reference's k = 10
        dict(name="reassign_4m", kind="reassign", ngroups=26, n_sub=50_000, k=10),
        # the classifier: loss gradient of a training set, and inference on it
        dict(name="classifier_400k", kind="mlp", n=400_003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["one", "batch", "batch", "batch", "learned", "resident", "tree", "direct", "reassign", "mlp"])
    bmp = rng.choice([0.995, 0.995, 1.0])
    if kind == "one":
        return dict(kind=kind, n=_log(rng, 60, 200_000), plain=rng.random() < 0.5, bmp=bmp)
    if kind == "batch":
        return dict(kind=kind, n=_log(rng, 20_000, 7_500_000), nmax=rng.choice([500, 2000, 50_000, 1_000_000]),
                    hydro=rng.random() < 0.35, defaults=rng.random() < 0.3, bmp=bmp)
    if kind == "learned":
        return dict(kind=kind, n=_log(rng, 100_000, 4_000_000), nmax=1_000_000,
                    min_particles=rng.choice([1000, 10_000, 30_000]), bmp=bmp)
    if kind == "resident":
        return dict(kind=kind, n=_log(rng, 30_000, 5_000_000), nmax=rng.choice([2000, 50_000, 1_000_000]), bmp=bmp)
    if kind == "tree":
        return dict(kind=kind, n=_log(rng, 5_000, 2_000_000), nsub=rng.randint(1, 50))
    if kind == "direct":
        return dict(kind=kind, n_src=_log(rng, 50, 60_000), n_tgt=_log(rng, 50, 60_000), periodic=rng.random() < 0.3)
    if kind == "reassign":
        return dict(kind=kind, ngroups=_log(rng, 2, 40), n_sub=_log(rng, 1000, 50_000), k=rng.choice([1, 5, 10, 10, 20, 32]))
    return dict(kind=kind, n=_log(rng, 3_000, 800_000))


def params(case):
    if case.get("defaults"):
        # hbtx_default_params, in a box
        return hbtx.workload_params(theta=0.45, max_sample_size=1000, refine_most_bound=1, periodic=1, box_size=50.0,
                                    direct_cutoff=-1, bound_mass_precision=case["bmp"],
                                    dm_only=0 if case.get("hydro") else 1, thermal=1 if case.get("hydro") else 0)
    return hbtx.workload_params(direct_cutoff=-1, bound_mass_precision=case.get("bmp", 0.995),
                                dm_only=0 if case.get("hydro") else 1, thermal=1 if case.get("hydro") else 0)


# --- inputs --------------------------------------------------------------------------

_XG = np.concatenate([[0.0], np.geomspace(1e-7, 64.0, 6000)])


def _mu(x):
    return np.log1p(x) - x / (1.0 + x)


class Drawer:
    """NFW particles on the GPU in double precision."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.xg = torch.from_numpy(_XG).cuda()
        self.mu = torch.from_numpy(_mu(_XG)).cuda()
        # Jeans integral of a profile truncated at x = 64 (synth.nfw_sigma2 in units of its prefactors)
        x = _XG[1:]
        j = synth.nfw_sigma2(x, 64.0, float(_mu(64.0)), 1.0) / (x * (1.0 + x) ** 2)
        self.jeans = torch.from_numpy(np.concatenate([[j[0]], j])).cuda()

    def rand(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda", dtype=torch.float64)

    def randn(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float64)

    def lookup(self, v, xs, ys):
        i = torch.searchsorted(xs, v.contiguous()).clamp(1, len(xs) - 1)
        x0, x1 = xs[i - 1], xs[i]
        return ys[i - 1] + (ys[i] - ys[i - 1]) * ((v - x0) / (x1 - x0)).clamp(0.0, 1.0)

    def mu_of(self, x):
        return torch.log1p(x) - x / (1.0 + x)

    def unit(self, n):
        z = 2.0 * self.rand(n) - 1.0
        phi = 2.0 * math.pi * self.rand(n)
        s = torch.sqrt((1.0 - z * z).clamp_min(0.0))
        return torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1)

    def sigma(self, x, c, gm, rs):
        x = torch.minimum(x, c)
        s2 = x * (1.0 + x) ** 2 * (self.lookup(x, self.xg, self.jeans) - self.lookup(c, self.xg, self.jeans)).clamp_min(0.0)
        return torch.sqrt(gm / (rs * self.mu_of(c)) * s2)

    def potential(self, x, c, gm, rs):
        xx = x.clamp_min(1e-12)
        inside = gm / (rs * self.mu_of(c)) * (self.mu_of(xx) / xx + 1.0 / (1.0 + x) - 1.0 / (1.0 + c))
        return -torch.where(x < c, inside, gm / (rs * xx))


def _population(seed, n, nmax, hydro=False, defaults=False, evolved=False, single=False):
    """A Population of exactly n particles: NFW subhaloes of [20, nmax] particles
    with dN/dN ~ N^-1.9, 10% interlopers (20% of a single halo).  evolved: the
    subhaloes after tidal stripping, and the previous snapshot's outputs."""
    rng = np.random.default_rng(seed)
    frac = 0.2 if single else 0.1
    if single:
        tot = np.array([n])
    else:
        tot, have = [], 0
        sizes = np.random.default_rng([n, nmax])  # (a case's subhaloes keep their sizes from seed to seed)
        while have < n:
            c = synth.draw_counts(sizes, 4096, 20, nmax, 1.9)
            c = c + np.floor(frac * c).astype(np.int64)
            tot.append(c)
            have += int(c.sum())
        tot = np.concatenate(tot)
        k = int(np.searchsorted(np.cumsum(tot), n))
        tot = tot[:k + 1]
        tot[k] -= int(tot.sum()) - n
    ninter = np.floor(tot * (frac / (1.0 + frac))).astype(np.int64)
    nmem = tot - ninter
    nsub = len(tot)
    box = 50.0
    conc = 10.0 ** rng.normal(math.log10(8.0), 0.15, nsub)
    r200 = synth.R200_PER_1E4 * np.cbrt(nmem / 1e4)
    rs = r200 / conc
    # (periodic: centres anywhere, so that subhaloes cross the box faces)
    centre = rng.uniform(0.0, box, (nsub, 3)) if defaults else rng.uniform(0.1 * box, 0.9 * box, (nsub, 3))
    bulk = rng.normal(0.0, 100.0, (nsub, 3))
    offsets = np.concatenate([[0], np.cumsum(tot)]).astype(np.int64)

    D = Drawer(seed)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    counts = dev(tot)
    sid = torch.repeat_interleave(torch.arange(nsub, device="cuda"), counts)
    local = torch.arange(n, device="cuda") - dev(offsets[:-1])[sid]
    inter = local >= dev(nmem)[sid]
    c, s = dev(conc)[sid], dev(rs)[sid]
    gm = synth.G_GRAV * MASS * dev(nmem.astype(np.float64))[sid]
    u = D.rand(n)
    x = torch.where(inter, 3.0 * c * u.pow(1.0 / 3.0), D.lookup(u * D.mu_of(c), D.mu, D.xg))
    phi = D.potential(x, c, gm, s)
    vesc = torch.sqrt(2.0 * phi.abs())
    dx = D.unit(n) * (x * s)[:, None]
    dv = D.randn(n, 3) * torch.where(inter, math.sqrt(3.0) * vesc, D.sigma(x, c, gm, s))[:, None]
    mass = torch.full((n,), MASS, device="cuda", dtype=torch.float64)
    ptype = u_int = None
    if hydro:
        d = D.rand(n)
        ptype = torch.where(d < 0.70, 1, torch.where(d < 0.90, 0, torch.where(d < 0.99, 4, 5)))
        xm = c.clamp_max(2.1626)
        vmax2 = gm / (s * D.mu_of(c)) * D.mu_of(xm) / xm
        u_int = torch.where(ptype == 0, 0.3 * vmax2 * torch.pow(10.0, 0.2 * D.randn(n)), torch.zeros_like(vmax2))
        bh = ptype == 5
        mass = torch.where(bh, 100.0 * mass, mass)
        dx = torch.where(bh[:, None], 0.1 * dx, dx)
    prev = None
    if evolved:
        # particles outside the tidal radius were kicked out: long ago beyond 0.9^5 r_200, just now beyond 0.9^6
        old = ~inter & (x > c * 0.9 ** 5)
        new = ~inter & ~old & (x > c * 0.9 ** 6)
        e_prev = 0.5 * dv.square().sum(1) + phi
        e_prev = torch.where(old, e_prev.abs() + vesc * vesc, e_prev)
        bound = e_prev < 0.0  # (a few interlopers are slow enough)
        prev = (bound, e_prev)
        kick = dv * (1.5 * vesc / dv.norm(dim=1).clamp_min(1e-6))[:, None]  # (along the velocity: unbound for good)
        dv = torch.where((old | new)[:, None], dv + kick, dv)
        dx = torch.where(old[:, None], dx + 0.004 * dv, dx) * (1.0 + 0.02 * D.randn(n, 3))
    pos, vel = dx + dev(centre)[sid], dv + dev(bulk)[sid]
    if defaults:
        pos = torch.remainder(pos, box)
        # subsampling takes the leading particles: the order in a subhalo is shuffled, black holes lead
        key = D.rand(n)
        if hydro:
            key = torch.where(ptype == 5, key - 2.0, key)
        o = torch.argsort(sid.double() * 4.0 + key, stable=True)
        pos, vel, mass = pos[o], vel[o], mass[o]
        ptype, u_int = (None, None) if not hydro else (ptype[o], u_int[o])
    f32 = lambda t: t.to(torch.float32).cpu().numpy()  # noqa: E731
    # the frames that the subhaloes had a snapshot ago: near their centres
    ref_pos = centre + rng.normal(0.0, 1.0, (nsub, 3)) * (0.02 * r200)[:, None]
    if defaults:
        ref_pos = np.mod(ref_pos, box)
    pop = synth.Population(f32(pos), f32(vel), f32(mass), offsets, np.arange(n, dtype=np.int64),
                           None if ptype is None else ptype.to(torch.int32).cpu().numpy(),
                           None if u_int is None else f32(u_int), ref_pos, bulk + rng.normal(0.0, 2.0, (nsub, 3)))
    if not evolved:
        return pop, None
    bound, e_prev = prev
    o = torch.argsort(e_prev + 1e12 * (~bound), stable=True)
    o = o[torch.argsort(sid[o], stable=True)]
    rank = torch.empty(n, dtype=torch.int64, device="cuda")
    rank[o] = local
    b = bound.cpu().numpy()
    nb = np.add.reduceat(b.astype(np.int64), offsets[:-1])
    r2 = np.add.reduceat((x * s).square().cpu().numpy() * b, offsets[:-1])
    return pop, dict(rank=rank.to(torch.int32).cpu().numpy(), bound=b.astype(np.uint8), energy=f32(e_prev),
                     com_pos=centre.astype(np.float32), com_vel=bulk.astype(np.float32),
                     mbound=(MASS * np.maximum(nb, 1)).astype(np.float32),
                     rscale=np.sqrt(r2 / np.maximum(nb, 1)).astype(np.float32))


def _host_haloes(seed, ngroups, n_sub):
    """synth.host_haloes with sizes that belong to the case: host haloes of 1 to 12
    NFW clumps of 50 to n_sub particles, 79% tracers, a fifth of the gas astray in
    another clump of its host."""
    sizes = np.random.default_rng([ngroups, n_sub])
    subs = sizes.integers(1, 13, ngroups)
    cnt = sizes.integers(50, n_sub + 1, int(subs.sum()))
    group = np.repeat(np.arange(ngroups), subs)
    first = np.concatenate([[0], np.cumsum(subs)])
    rng = np.random.default_rng(seed)
    host = rng.uniform(0.5, 1.5, (ngroups, 3)) + 3.0 * np.arange(ngroups)[:, None]
    inner = (np.arange(len(cnt)) > first[group])[:, None]
    centre = host[group] + rng.normal(0.0, 0.05, (len(cnt), 3)) * inner
    scale = 0.02 * (cnt / np.maximum.reduceat(cnt, first[:-1])[group]) ** (1 / 3) + 1e-3
    n = int(cnt.sum())
    D = Drawer(seed)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    sub = torch.repeat_interleave(torch.arange(len(cnt), device="cuda"), dev(cnt))
    tracer = D.rand(n) < 0.79
    ns, f = dev(subs[group])[sub], dev(first[group])[sub]
    astray = ~tracer & (D.rand(n) < 0.2) & (ns > 1)
    step = 1 + (D.rand(n) * (ns - 1)).long().clamp_max(10)
    clump = torch.where(astray, f + (sub - f + step) % ns, sub)
    c = torch.full((n,), 10.0, device="cuda", dtype=torch.float64)
    x = D.lookup(D.rand(n) * D.mu_of(c), D.mu, D.xg) * dev(scale)[clump]
    pos = D.unit(n) * x[:, None] + dev(centre)[clump]
    goff = np.concatenate([[0], np.cumsum(cnt)])[first].astype(np.int64)
    return synth.HostHalos(pos.to(torch.float32).cpu().numpy(), tracer.to(torch.uint8).cpu().numpy(),
                           sub.to(torch.int32).cpu().numpy(), goff, None)


def _weights(seed):
    """Network weights: the initialisation's scale, with one unit of each layer
    carrying the previous bound flag to the logit (as training ends up doing)."""
    rng = np.random.default_rng([seed, 7])
    w = np.zeros(hbtx.MLP_NPAR, np.float32)
    p = hbtx.mlp_unpack(w)
    p["W1"][:] = rng.uniform(-0.05, 0.05, (64, 8))
    p["W2"][:] = rng.uniform(-0.05, 0.05, (64, 64))
    p["w3"][:] = rng.uniform(-0.05, 0.05, 64)
    p["W1"][0] = 0.0
    p["W1"][0, 3] = 1.0
    p["W2"][0] = 0.0
    p["W2"][0, 0] = 1.0
    p["w3"][0] = 12.0
    p["b3"][:] = -7.0
    return w


def _samples(seed, n):
    """Feature rows of the ranges that the previous snapshot's outputs give, and bound flags."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    r = torch.rand(n, 8, generator=g, device="cuda")
    bound = (r[:, 3] < 0.6).float()
    X = torch.stack([3.0 * r[:, 0] - 2.0, 4.0 * r[:, 1] * r[:, 1], r[:, 2], bound, 0.2 + 0.0 * r[:, 4],
                     -6.0 * r[:, 5], 0.2 + 0.8 * r[:, 6], -4.0 * r[:, 7] + 2.0 * (1.0 - bound)], 1)
    y = (bound > 0) ^ (r[:, 4] < 0.05)
    return X.cpu().numpy(), y.to(torch.uint8).cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind)
    if kind in ("one", "batch", "resident"):
        st["prm"] = params(case)
        st["pop"], _ = _population(seed, case["n"], case.get("nmax", 0), case.get("hydro", False),
                                   case.get("defaults", False), single=kind == "one")
        st["flags"] = hbtx.PLAIN if case.get("plain") else hbtx.BATCHED
        if kind == "resident":
            st["ctx"] = hbtx.Context(0)
            st["ctx"].load(st["pop"])
    elif kind == "learned":
        st["prm"] = params(case)
        st["min_particles"] = case["min_particles"]
        st["pop"], st["prev"] = _population(seed, case["n"], case["nmax"], evolved=True)
        st["net"] = hbtx.MLP(context(), 0)
        st["net"].set_weights(_weights(seed))
    elif kind == "tree":
        h = _population(seed, case["n"], 0, single=True)[0]
        # embedded subhaloes: equal shares of a tenth of the particles, compact, around points of the host
        rng = np.random.default_rng(seed)
        m = case["n"] // 10 // case["nsub"]
        for k in range(case["nsub"] if m > 1 else 0):
            sl = slice(k * m, (k + 1) * m)
            at = h.pos[rng.integers(0, case["n"])].copy()
            h.pos[sl] = at + 0.05 * (h.pos[sl] - h.pos[sl].mean(0))
        st["prm"] = params(case)
        st["pos"], st["mass"] = h.pos, h.mass
    elif kind == "direct":
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        ns, nt = case["n_src"], case["n_tgt"]
        # sources of one halo, some across the box face where periodic; half of the targets are sources
        centre = 0.02 if case["periodic"] else 2.0
        src = (0.05 * torch.randn(ns, 3, generator=g, device="cuda") + centre)
        st["mass"] = 0.01 * (0.5 + 1.5 * torch.rand(ns, generator=g, device="cuda"))
        tgt = (0.08 * torch.randn(nt, 3, generator=g, device="cuda") + centre)
        if case["periodic"]:
            src, tgt = torch.remainder(src, 4.0), torch.remainder(tgt, 4.0)
        tm = torch.zeros(nt, device="cuda")
        k = min(ns, nt // 2)
        tgt[:k], tm[:k] = src[:k], st["mass"][:k]
        st["src"], st["tgt"], st["tm"] = src.contiguous(), tgt.contiguous(), tm
        st["out"] = torch.zeros(nt, device="cuda", dtype=torch.float64)
        st["prm"] = hbtx.make_params(**_direct_params(case))
        context()
    elif kind == "reassign":
        st["h"] = _host_haloes(seed, case["ngroups"], case["n_sub"])
        st["k"] = case["k"]
        st["prm"] = params(case)
    else:
        st["X"], st["y"] = _samples(seed, case["n"])
        st["net"] = hbtx.MLP(context(), 0)
        st["net"].set_weights(_weights(seed))
    context()
    return st


def _direct_params(case):
    return hbtx.workload_params(**(dict(periodic=1, box_size=4.0) if case["periodic"] else {}))


# --- one pass ------------------------------------------------------------------------

def _outputs(out):
    r = dict(order=out["order"], energy=out["energy"], result={k: out["result"][k] for k in hbtx.RESULT_DTYPE.names})
    if out["potential"] is not None:
        r["potential"] = out["potential"]
    return r


def run(st):
    kind, ctx = st["kind"], context()
    if kind in ("one", "batch"):
        return _outputs(ctx.unbind(st["pop"], st["prm"], st["flags"]))
    if kind == "resident":
        c = st["ctx"]
        c.run(st["prm"], hbtx.SAVE_POTENTIAL)
        prof = c.profiles(st["prm"])
        r = _outputs(c.fetch(want_potential=True))
        r["profiles"] = {k: prof[k] for k in hbtx.PROFILE_DTYPE.names if k != "reserved"}
        return r
    if kind == "learned":
        return _outputs(learned.warm_unbind(ctx, st["pop"], st["prev"], st["net"], st["prm"],
                                            min_particles=st["min_particles"])[0])
    if kind == "tree":
        tree = ctx.tree(st["pos"], st["mass"], st["prm"])
        phi = tree.potential(st["pos"], st["mass"])
        tree.close()
        return phi
    if kind == "direct":
        ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        rc = hbtx.lib().hbtx_direct_potential_noalloc(ctx._h, ctypes.byref(st["prm"]), len(st["src"]), ptr(st["src"]),
                                                      ptr(st["mass"]), len(st["tgt"]), ptr(st["tgt"]), ptr(st["tm"]),
                                                      ptr(st["out"]))
        if rc != hbtx.OK:
            raise hbtx.HbtxError(rc, "hbtx_direct_potential_noalloc")
        return st["out"]
    if kind == "reassign":
        h = st["h"]
        return ctx.reassign_targets(h.pos, h.is_tracer, h.sub, h.group_offsets, k=st["k"], params=st["prm"])[0]
    grad, loss = st["net"].gradient(st["X"], st["y"])
    return dict(grad=grad, loss=loss, logit=st["net"].predict(st["X"]))


# --- what a pass cannot do without -----------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("one", "batch", "learned", "resident"):
        n = case["n"]
        per_in = 28 + 8 + (8 if case.get("hydro") else 0)  # positions, velocities, masses, ids (types, energies)
        if kind == "resident":
            per_in = 32
        if kind == "learned":
            per_in += 9
        # one evaluation of every particle's potential: about 200 records of 16 flops a target (theta = 0.7)
        pairs = min(n, 200)
        return dict(bytes=float(n * (per_in + 12 + (4 if kind == "resident" else 0))), flops=float(n * pairs * 16))
    if kind == "tree":
        return dict(bytes=float(case["n"] * (16 + 16 + 8)), flops=float(case["n"] * 200 * 16))
    if kind == "direct":
        return dict(bytes=float(16 * case["n_src"] + 24 * case["n_tgt"]), flops=14.0 * case["n_src"] * case["n_tgt"])
    if kind == "reassign":
        n = case["ngroups"] * 6.5 * case["n_sub"] / 2
        return dict(bytes=float(n * 21), flops=float(0.21 * n * 10 * max(2 * case["k"], 32)))
    return dict(bytes=float(case["n"] * (2 * 32 + 1 + 4)), flops=float(case["n"] * (3 + 1) * 2 * 4672))


# --- 64-bit values -----------------------------------------------------------------------

def exact(case, seed):
    """The exact sum and the classifier in double precision (the unbinding's tree
    approximation and its integer decisions have no such value)."""
    if case["kind"] == "direct":
        return _exact_direct(case, seed)
    if case["kind"] == "mlp":
        return _exact_mlp(case, seed)
    return None


def _exact_direct(case, seed):
    st = prepare(case, seed)
    p = _direct_params(case)
    src, m, tgt, tm = (st[k].double() for k in ("src", "mass", "tgt", "tm"))
    eps = float(np.float32(p["softening"]))
    h = float(np.float32(2.8 * eps))
    out = torch.empty(len(tgt), device="cuda", dtype=torch.float64)
    for a in range(0, len(tgt), 1024):
        d = tgt[a:a + 1024, None, :] - src[None, :, :]
        if case["periodic"]:
            d = torch.where(d > 2.0, d - 4.0, torch.where(d < -2.0, d + 4.0, d))
        r = torch.sqrt(d.square().sum(2))
        u = r / h
        near = torch.where(u < 0.5, -2.8 + u * u * (16.0 / 3.0 + u * u * (6.4 * u - 9.6)),
                           -3.2 + 1.0 / (15.0 * u.clamp_min(1e-30))
                           + u * u * (32.0 / 3.0 + u * (-16.0 + u * (9.6 - 32.0 / 15.0 * u)))) / h
        phi = torch.where(u < 1.0, near, -1.0 / r.clamp_min(1e-30))
        out[a:a + 1024] = ((phi * m[None, :]).sum(1) + tm[a:a + 1024] / eps) * p["G"]
    return out


def _exact_mlp(case, seed):
    X, y = _samples(seed, case["n"])
    w = torch.from_numpy(_weights(seed)).cuda().to(torch.bfloat16).double()
    W1, b1, W2, b2 = w[:512].view(64, 8), w[512:576], w[576:4672].view(64, 64), w[4672:4736]
    w3, b3 = w[4736:4800], w[4800]
    grad = torch.zeros_like(w)
    logits, loss, n = [], 0.0, len(X)
    for a in range(0, n, 1 << 18):
        x = torch.from_numpy(X[a:a + (1 << 18)]).cuda().double()
        t = torch.from_numpy(y[a:a + (1 << 18)]).cuda().double()
        h1 = torch.relu(x @ W1.T + b1)
        h2 = torch.relu(h1 @ W2.T + b2)
        z = h2 @ w3 + b3
        logits.append(z)
        loss += float((torch.nn.functional.softplus(z) - t * z).sum())
        dz = (torch.sigmoid(z) - t) / n
        d2 = dz[:, None] * w3[None, :] * (h2 > 0)
        d1 = (d2 @ W2) * (h1 > 0)
        grad += torch.cat([(d1.T @ x).reshape(-1), d1.sum(0), (d2.T @ h1).reshape(-1), d2.sum(0), h2.T @ dz,
                           dz.sum().reshape(1)])
    return dict(grad=grad, loss=loss / n, logit=torch.cat(logits))
