"""What this library is measured on: the work a simulation program has it do,
through the package's public entry points.

Three kinds of case:
  step      one system advanced by the number of steps between two outputs,
            then what that output needs read back (positions; on the FP64
            path also the bond forces and tensions; with thermodynamics on,
            the pressure and the bond energies)
  serve     a batch of independent systems handed to the ensemble runner and
            drained, the final positions read back
  analyse   one sample of the on-device analyses of a system
A system is a periodic tile of randomly inserted filaments (the package's own
generator), repeated tiles x tiles x tiles times, which gives large systems
of the same density, length and stiffness distributions quickly.
"""
import ctypes
import math

import numpy as np
import torch

import simcore_amd as sc
from simcore_amd import workloads
from simcore_amd._lib import ScFilamentParams

DELTA = {"dense": 1e-4, "uneven": 1e-5, "long": 1e-5}
XLINK = dict(k_spring=10.0, rest_length=1.0, k_off=0.1, r_bind=2.0, seed=14)


def _case(name, kind, system, filaments, tiles, sites, precision, steps, **kw):
    c = {"kind": kind, "system": system, "filaments": filaments, "tiles": tiles, "sites": sites,
         "precision": precision, "steps": steps, "graph": True, "order": True, "tuned": False,
         "crosslinks": 0, "thermo": False}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the parity configuration (64 filaments x 20 sites, FP64, plain
        # launches) as a plugin of the reference drives it: one time step,
        # that is a midstep and a full step, and its state read back
        _case("parity_one_step", "step", "dense", 64, 1, 20, "fp64", 2, graph=False, order=False),
        # a small system of a parameter scan, alone on the device
        _case("small_1k", "step", "dense", 32, 1, 32, "mixed", 50),
        # a system of ordinary size with an odd filament length
        _case("ordinary_52k", "step", "dense", 1999, 1, 27, "mixed", 50),
        # the dense single system of the benchmark, at its launch shape
        _case("dense_620k", "step", "dense", 2500, 2, 32, "mixed", 100, tuned=True),
        # the uneven-length system of the benchmark (its default workload)
        _case("uneven_1600k", "step", "uneven", 1852, 3, 0, "mixed", 100, tuned=True),
        # its crosslinked variant, a quarter of the size
        _case("crosslinked_400k", "step", "uneven", 1563, 2, 0, "mixed", 50, crosslinks=50000),
        # filaments of 129-256 sites only
        _case("long_110k", "step", "long", 70, 2, 256, "mixed", 50),
        # the bit-exact path, which validation runs and plain callers take
        _case("exact_dense_155k", "step", "dense", 625, 2, 32, "fp64", 20, order=False),
        _case("exact_uneven_230k", "step", "uneven", 925, 2, 0, "fp64", 20, order=False),
        # a run with thermodynamic output
        _case("thermo_62k", "step", "dense", 250, 2, 32, "mixed", 50, thermo=True),
        # systems of 1k-100k bonds handed to the ensemble runner at once
        _case("serve_24", "serve", "dense", 24, 1, 32, "mixed", 200),
        # one sample of the mse2e and theta analyses of the dense system
        _case("analyse_620k", "analyse", "dense", 2500, 2, 32, "mixed", 0),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "dense", "dense", "uneven", "uneven", "long", "exact", "exact",
                       "crosslinked", "thermo", "serve", "analyse"])
    steps = 2 * rng.randint(10, 25) + rng.randint(0, 1)
    order = rng.random() < 0.8
    if kind == "small":
        return _case("", "step", "dense", rng.randint(16, 200), 1, rng.randint(8, 33),
                     rng.choice(["mixed", "fp64"]), rng.choice([1, 2, 9, steps]),
                     graph=rng.random() < 0.5, order=False)
    if kind == "dense":
        return _case("", "step", "dense", _log_uniform(rng, 200, 2000), rng.choice([1, 2]),
                     rng.randint(3, 33), "mixed", steps, order=order, tuned=rng.random() < 0.5)
    if kind == "uneven":
        return _case("", "step", "uneven", _log_uniform(rng, 300, 1500), rng.choice([1, 2, 3]), 0,
                     "mixed", steps, order=order, tuned=rng.random() < 0.5)
    if kind == "long":
        return _case("", "step", "long", rng.randint(20, 70), rng.choice([1, 2]),
                     rng.randint(140, 256), "mixed", steps, order=order)
    if kind == "exact":
        if rng.random() < 0.5:
            return _case("", "step", "dense", _log_uniform(rng, 40, 700), rng.choice([1, 2]),
                         rng.randint(3, 33), "fp64", steps // 2, order=False,
                         graph=rng.random() < 0.7)
        return _case("", "step", "uneven", _log_uniform(rng, 250, 900), rng.choice([1, 2]), 0,
                     "fp64", steps // 2, order=False, graph=rng.random() < 0.7)
    if kind == "crosslinked":
        return _case("", "step", "uneven", _log_uniform(rng, 300, 1500), rng.choice([1, 2]), 0,
                     rng.choice(["mixed", "mixed", "fp64"]), steps, order=order,
                     crosslinks=_log_uniform(rng, 2000, 50000))
    if kind == "thermo":
        return _case("", "step", "dense", _log_uniform(rng, 100, 1000), rng.choice([1, 2]),
                     rng.randint(8, 33), rng.choice(["mixed", "mixed", "fp64"]), steps,
                     order=order, thermo=True)
    if kind == "serve":
        return _case("", "serve", "dense", rng.randint(4, 24), 1, rng.randint(12, 32), "mixed",
                     2 * rng.randint(25, 100))
    return _case("", "analyse", rng.choice(["dense", "uneven"]), _log_uniform(rng, 300, 1500),
                 rng.choice([1, 2]), rng.randint(8, 32), rng.choice(["mixed", "fp64"]), 0,
                 order=order)


# ---------------------------------------------------------------- inputs ----

def _tile(case, seed):
    """(params, filaments) of one tile."""
    kind, nf, n = case["system"], case["filaments"], case["sites"]
    delta = DELTA[kind]
    if kind == "dense":
        p, fil, _ = workloads.dense(nf=nf, n_sites=n, seed=seed + 1, delta=delta)
    elif kind == "uneven":
        # the lengths are the case's, the positions the seed's
        p, fil, _ = workloads.uneven(nf=nf, rng_seed=nf, seed=seed + 1, delta=delta)
    else:
        rng = np.random.default_rng(nf)
        sites = rng.integers(129, n + 1, nf)
        R = workloads.box_for_fraction(sites, 1.0, 1.0, 0.02)
        p = sc.params_init(R, delta=delta, min_cell_length=1.0)
        fil = sc.generate_filaments(p, sites, (sites - 1).astype(float),
                                    rng.uniform(10.0, 1000.0, nf), 1.0, 2.0, seed=seed + 1)
    return p, fil


def _repeat(p, fil, t, noise_seed):
    """The tile repeated t times along each axis, with its noise stream."""
    if t > 1:
        side, nt = 2.0 * p.system_radius, t ** 3
        shift = side * np.stack(np.meshgrid(*[np.arange(t)] * 3, indexing="ij"), -1).reshape(-1, 3)
        shift -= 0.5 * side * (t - 1)
        big = (fil.r.reshape(3, 1, -1) + shift.T[:, :, None]).reshape(-1)
        off = (fil.site_off[None, :-1] + fil.ns * np.arange(nt)[:, None]).reshape(-1)
        par = (ScFilamentParams * (fil.nf * nt))()
        one = bytes(fil.fil)
        ctypes.memmove(par, one * nt, len(one) * nt)
        fil = sc.Filaments(np.append(off, fil.ns * nt).astype(np.int32),
                           np.ascontiguousarray(big), par)
        p = sc.params_init(t * p.system_radius, delta=p.delta, min_cell_length=1.0)
    p.seed = noise_seed
    return p, fil


def _system(case, seed):
    """(params, filaments) of a case."""
    p, fil = _tile(case, seed)
    return _repeat(p, fil, case["tiles"], 1000003 * (seed + 1))


def _crosslinks(case, seed, p, fil):
    return sc.generate_crosslinks(p, fil, case["crosslinks"], r_bind=2.0, seed=seed + 2)


def _requests(case, seed):
    """(params, filaments) of every system of a serving batch: 1k-100k bonds,
    spread evenly over their logarithm, persistence lengths U[10, 1000]."""
    rng = np.random.default_rng(seed)
    n, out = case["sites"], []
    for k in range(case["filaments"]):
        nb = 1e3 * 100.0 ** ((k + 0.5) / case["filaments"])
        nf = max(1, int(round(nb / (n - 1))))
        t = 2 if nf >= 400 else 1
        sub = dict(case, filaments=max(1, nf // t ** 3), tiles=t)
        R = workloads.box_for_fraction([n] * sub["filaments"], 1.0, 1.0, 0.05)
        p = sc.params_init(R, delta=1e-5, min_cell_length=1.0)
        fil = sc.generate_filaments(p, [n] * sub["filaments"], n - 1.0, rng.uniform(10.0, 1000.0),
                                    1.0, 2.0, seed=int(rng.integers(1, 2 ** 31)))
        out.append(_repeat(p, fil, t, int(rng.integers(1, 2 ** 62))))
    return out


def prepare(case, seed):
    if case["kind"] == "serve":
        return {"case": case, "requests": _requests(case, seed),
                "runner": sc.Ensemble(hbm_budget=8 << 30, max_active=64, steps_per_launch=64,
                                      batch_size=16)}
    p, fil = _system(case, seed)
    s = sc.FilamentSystem(p, fil, precision=case["precision"], use_graph=case["graph"],
                          spatial_order=case["order"])
    if case["crosslinks"]:
        s.load_crosslinks(*_crosslinks(case, seed, p, fil), **XLINK)
    if case["tuned"]:  # the benchmark's fixed launch shape
        s.set_launch_shape(0, 1, 2, 2, 0)
    if case["thermo"]:
        s.thermo_enable()
    return {"case": case, "system": s, "r": np.empty(3 * fil.ns)}


def run(state):
    case = state["case"]
    if case["kind"] == "serve":
        runner = state["runner"]
        ids = [runner.submit(p, f, case["steps"], precision=case["precision"],
                             spatial_order=case["order"]) for p, f in state["requests"]]
        runner.drain()
        return [runner.result(i) for i in ids]
    s = state["system"]
    if case["kind"] == "analyse":
        e2e, com = s.filament_stats()
        return {"e2e": e2e, "com": com, "theta": s.theta_histogram(100, 31)}
    s.step(case["steps"])
    if case["precision"] == "fp64" and not case["crosslinks"]:
        r, r_prev, f_rand = s.sites()
        f, t = s.bond_forces()
        out = {"r": r, "r_prev": r_prev, "f_rand": f_rand, "force": f, "torque": t,
               "tension": s.tensions()}
    else:
        # the positions alone, into the caller's mirror
        r = state["r"]
        rc = sc.lib.sc_get_sites(s.h, r.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), None,
                                 None)
        if rc:
            raise sc.SimcoreError(rc, "sc_get_sites")
        out = {"r": r}
    if case["thermo"]:
        out.update(s.calculate_pressure(case["steps"]), energy=s.bond_energies())
    return out


# ---------------------------------------------------------------- bounds ----

def _sizes(case):
    """(filaments, sites) expected of a case's system."""
    t3 = case["tiles"] ** 3
    nf = case["filaments"] * t3
    per = {"dense": case["sites"], "uneven": 31.7, "long": 0.5 * (129 + case["sites"])}
    return nf, nf * per[case["system"]]


def work(case):
    """Bytes and operations of a pass: per step each state array read and
    written once (per bond its record read, its force and torque written and
    read, its new record written; per site the position read and written,
    the midstep start, the random force and the displacement bookkeeping;
    per candidate pair its two entries and slots), then the results read."""
    mixed = case["precision"] == "mixed"
    rec, sums, slot = (32, 24, 16) if mixed else (64, 48, 32)
    if case["kind"] == "serve":
        nb = sum(1e3 * 100.0 ** ((k + 0.5) / case["filaments"]) for k in range(case["filaments"]))
        nf = nb / (case["sites"] - 1)
        ns = nb + nf
    else:
        nf, ns = _sizes(case)
        nb = ns - nf
    if case["kind"] == "analyse":
        return {"bytes": 24 * ns + rec * nb + 48 * nf + 8 * 3100, "flops": 3 * ns + 8 * nb}
    nc = (1.45 if case["system"] == "uneven" else 0.9) * nb
    per_step = nb * (2 * rec + 2 * sums + 4) + nc * 2 * (slot + 8) + ns * 148
    if not mixed:
        per_step += ns * 24
    ops = nc * 2 * 150 + ns * 1200
    if case["crosslinks"]:
        per_step += case["crosslinks"] * (72 + 24)
        ops += case["crosslinks"] * 100
    out = 24 * ns if mixed or case["crosslinks"] else 72 * ns + 56 * nb
    if case["thermo"]:
        out += 8 * nb
    return {"bytes": case["steps"] * per_step + out, "flops": case["steps"] * ops}


# ----------------------------------------------------- plain FP64 results ----
# The model in plain torch, vectorised over bonds, pairs and filaments, with
# none of the library's code: the reference's filament step (cell-list
# candidates with sticky forces, WCA pairs, random forces projected onto the
# constraints, bending with the metric correction, constraint tensions,
# midstep integration, renormalisation).

def _mul32(a, b):
    """(high, low) 32 bits of the product of int64 tensor a < 2^32 and b < 2^32."""
    lo, hi = b & 0xFFFF, b >> 16
    high = (a * hi + ((a * lo) >> 16)) >> 16
    return high, ((a * lo) + (((a * hi) & 0xFFFF) << 16)) & 0xFFFFFFFF


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors of 32-bit words."""
    M = 0xFFFFFFFF
    for _ in range(10):
        h0, l0 = _mul32(c0, 0xD2511F53)
        h1, l1 = _mul32(c2, 0xCD9E8D57)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
    return c0, c1, c2, c3


def _dot(a, b):
    return (a * b).sum(-1)


class _Model:
    def __init__(self, p, fil, dev):
        self.p, self.dev = p, dev
        T = lambda x, t=torch.float64: torch.as_tensor(np.asarray(x), dtype=t, device=dev)  # noqa: E731
        off = np.asarray(fil.site_off, dtype=np.int64)
        n = np.diff(off)
        self.nf, self.ns, self.nb = fil.nf, fil.ns, fil.nb
        par = np.frombuffer(bytes(fil.fil), dtype=np.float64).reshape(-1, 5)
        self.box = 2.0 * p.system_radius
        rcut = 2.0 ** (1.0 / 6.0) * p.wca_sig
        self.rcut2 = rcut * rcut
        self.n1 = max(3, int(math.floor(self.box / max(p.min_cell_length, rcut))))
        self.thr = 0.25 * (self.box / self.n1) ** 2
        self.c12 = 4.0 * p.wca_eps * p.wca_sig ** 12
        self.c6 = 4.0 * p.wca_eps * p.wca_sig ** 6
        self.r = T(fil.r).reshape(3, -1).T.contiguous()
        self.rp, self.fr = self.r.clone(), torch.zeros_like(self.r)
        self.dr0 = self.r.clone()
        self.acc = torch.zeros(self.ns, dtype=torch.float64, device=dev)
        bf = np.repeat(np.arange(fil.nf), n - 1)
        self.bond_fil = T(bf, torch.int64)
        self.site0 = torch.arange(self.nb, device=dev) + self.bond_fil
        self.bl_bond = T(par[bf, 0])
        self.switch = torch.ones(self.nf, dtype=torch.bool, device=dev)
        self.k, self.drmax = 0, 0.0
        self.stress = torch.zeros(3, 3, dtype=torch.float64, device=dev)
        # filaments of like length, padded to one width
        self.groups = []
        lo = 0
        for hi in (8, 16, 32, 64, 128, 256):
            f = np.nonzero((n > lo) & (n <= hi))[0]
            lo = hi
            if not len(f):
                continue
            L = int(n[f].max())
            i = np.arange(L)[None, :]
            ok = i < n[f][:, None]
            self.groups.append({
                "f": T(f, torch.int64), "n": T(n[f], torch.int64)[:, None], "L": L,
                "site": T(np.where(ok, off[f][:, None] + i, off[f][:, None]), torch.int64),
                "ok": T(ok, torch.bool), "i": T(i, torch.int64),
                "bond": T((off[f] - f)[:, None] + np.minimum(i, (n[f] - 2)[:, None]), torch.int64),
                "bl": T(par[f, 0])[:, None], "kappa": T(par[f, 1])[:, None],
                "gpar": T(par[f, 2])[:, None], "gperp": T(par[f, 3])[:, None]})
        self.nx = 0
        self._bonds()
        self._rebuild()

    def crosslinks(self, bonds, lam):
        T = lambda x, t: torch.as_tensor(np.asarray(x), dtype=t, device=self.dev)  # noqa: E731
        self.xb, self.xl = T(bonds, torch.int64), T(lam, torch.float64)
        self.nx = len(self.xb)
        self.xF = torch.zeros(self.nx, 3, dtype=torch.float64, device=self.dev)
        self.xT = torch.zeros(self.nx, 2, 3, dtype=torch.float64, device=self.dev)

    def _wrap(self, d):
        return d - self.box * torch.round(d / self.box)

    def _bonds(self):
        o = self.r[self.site0 + 1] - self.r[self.site0]
        self.len = o.norm(dim=1)
        self.u = o / self.len[:, None]
        self.c = self.r[self.site0] + 0.5 * o

    def _rebuild(self):
        n = self.n1
        s = self.c / self.box
        s = s - torch.round(s)
        c = torch.clamp(torch.floor(n * (s + 0.5)).to(torch.int64), 0, n - 1)
        key = (c[:, 0] * n + c[:, 1]) * n + c[:, 2]
        ks, order = torch.sort(key, stable=True)
        a_all, b_all = [], []
        cells = [(0, 0, 0), (1, 0, 0), (-1, 1, 0), (0, 1, 0), (1, 1, 0)]
        cells += [(x, y, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
        cs = c[order]
        for d in cells:
            m = (cs + torch.tensor(d, device=self.dev)) % n
            kk = (m[:, 0] * n + m[:, 1]) * n + m[:, 2]
            lo, hi = torch.searchsorted(ks, kk), torch.searchsorted(ks, kk, right=True)
            if d == (0, 0, 0):
                lo = torch.arange(self.nb, device=self.dev) + 1
            cnt = torch.clamp(hi - lo, min=0)
            i = torch.repeat_interleave(torch.arange(self.nb, device=self.dev), cnt)
            first = torch.cumsum(cnt, 0) - cnt
            j = torch.arange(len(i), device=self.dev) - first[i] + lo[i]
            a_all.append(order[i])
            b_all.append(order[j])
        a, b = torch.cat(a_all), torch.cat(b_all)
        near = ((a - b).abs() == 1) & (self.bond_fil[a] == self.bond_fil[b])
        self.a, self.b = a[~near], b[~near]
        self.slot = torch.zeros(len(self.a), 3, dtype=torch.float64, device=self.dev)
        self.rs = torch.zeros(len(self.a), dtype=torch.float64, device=self.dev)
        self.dr0, self.acc = self.r.clone(), torch.zeros_like(self.acc)

    def _pairs(self, thermo):
        a, b, p = self.a, self.b, self.p
        dr = self._wrap(self.c[b] - self.c[a])
        u1, u2, h1, h2 = self.u[a], self.u[b], 0.5 * self.len[a], 0.5 * self.len[b]
        x, y, c = _dot(dr, u1), _dot(dr, u2), _dot(u1, u2)
        den = 1.0 - c * c
        flat = den < 1e-12
        den = torch.where(flat, torch.ones_like(den), den)
        la = torch.where(flat, 0.5 * x, (x - c * y) / den)
        mu = torch.where(flat, -0.5 * y, (-y + c * x) / den)
        clamp = lambda v, h: torch.minimum(torch.maximum(v, -h), h)  # noqa: E731
        end = lambda v, h: torch.where(v >= 0, h, -h)  # noqa: E731
        o1, o2 = la.abs() > h1, mu.abs() > h2
        la1 = end(la, h1)
        mu1 = clamp(-y + la1 * c, h2)
        mu2 = end(mu, h2)
        la2 = clamp(x + mu2 * c, h1)
        dist = lambda l, m: dr - l[:, None] * u1 + m[:, None] * u2  # noqa: E731
        use1 = o1 & (~o2 | (_dot(dist(la1, mu1), dist(la1, mu1)) <
                            _dot(dist(la2, mu2), dist(la2, mu2))))
        use2 = o2 & ~use1
        la = torch.where(use1, la1, torch.where(use2, la2, la))
        mu = torch.where(use1, mu1, torch.where(use2, mu2, mu))
        d = dist(la, mu)
        d2 = _dot(d, d)
        hit = d2 <= self.rcut2
        rm = torch.sqrt(d2)
        ri = 1.0 / rm
        r6 = ri ** 6
        ff = -(12.0 * self.c12 * r6 - 6.0 * self.c6) * r6 * ri
        ff = torch.clamp(ff, -p.f_cutoff, p.f_cutoff)
        self.slot = torch.where(hit[:, None], (ff * ri)[:, None] * d, self.slot)
        self.rs = torch.where(hit, rm, self.rs)
        F = torch.zeros(self.nb, 3, dtype=torch.float64, device=self.dev)
        Tq = torch.zeros_like(F)
        if self.nx:
            for q, s in ((0, 1.0), (1, -1.0)):
                F.index_add_(0, self.xb[:, q], s * self.xF)
                Tq.index_add_(0, self.xb[:, q], self.xT[:, q])
        F.index_add_(0, a, self.slot)
        F.index_add_(0, b, -self.slot)
        Tq.index_add_(0, a, torch.cross(la[:, None] * u1, self.slot, dim=1))
        Tq.index_add_(0, b, -torch.cross(mu[:, None] * u2, self.slot, dim=1))
        self.F, self.Tq = F, Tq
        if thermo:
            f1 = self.slot.norm(dim=1)
            w = torch.where(f1 > 0, self.rs / torch.where(f1 > 0, f1, torch.ones_like(f1)),
                            torch.zeros_like(f1))
            self.stress += (w[:, None] * self.slot).T @ self.slot
            on = self.rs > 0
            q6 = torch.where(on, 1.0 / torch.where(on, self.rs, torch.ones_like(self.rs)),
                             torch.zeros_like(self.rs)) ** 6
            e = torch.where(on, q6 * (self.c12 * q6 - self.c6) + p.wca_eps,
                            torch.zeros_like(q6))
            self.E = torch.zeros(self.nb, dtype=torch.float64, device=self.dev)
            self.E.index_add_(0, a, e)
            self.E.index_add_(0, b, e)

    def _anchor(self, bond, lam):
        u = self.u[bond]
        return self.c[bond] - ((0.5 * self.len[bond] - lam)[:, None]) * u

    def _springs(self):
        P = [self._anchor(self.xb[:, q], self.xl[:, q]) for q in (0, 1)]
        dr = self._wrap(P[1] - P[0])
        length = dr.norm(dim=1)
        self.xF = (XLINK["k_spring"] * (length - XLINK["rest_length"]) / length)[:, None] * dr
        for q, s in ((0, 1.0), (1, -1.0)):
            arm = (self.xl[:, q] - 0.5 * self.len[self.xb[:, q]])[:, None] * self.u[self.xb[:, q]]
            self.xT[:, q] = torch.cross(arm, s * self.xF, dim=1)

    def _rebind(self):
        m, dev = self.k // 2, self.dev
        prob = 1.0 - math.exp(-XLINK["k_off"] * self.p.delta)
        x = torch.arange(self.nx, device=dev)
        k0, k1 = XLINK["seed"] & 0xFFFFFFFF, XLINK["seed"] >> 32
        o = _philox(x, x * 0, x * 0 + m, x * 0 + 1, k0, k1)
        un = [(v.to(torch.float64) + 0.5) / 4294967296.0 for v in o]
        for i in torch.nonzero(un[0] < prob).ravel().tolist():
            moving = 0 if float(un[1][i]) < 0.5 else 1
            stay = self.xb[i, 1 - moving][None]
            P = self._anchor(stay, self.xl[i, 1 - moving][None])
            d = self._wrap(self.c - P)
            t = torch.minimum(torch.maximum(_dot(d, self.u), -0.5 * self.len), 0.5 * self.len)
            e = d - t[:, None] * self.u
            near = _dot(e, e) <= XLINK["r_bind"] ** 2
            near[stay] = False
            cand = torch.nonzero(near).ravel()
            if not len(cand):
                continue
            z = cand * 0
            score = _philox(z + i, z + m, cand, z + 2, k0, k1)[0]
            best = cand[torch.argmin(score * (1 << 31) + cand)]
            self.xb[i, moving] = best
            self.xl[i, moving] = un[2][i] * self.bl_bond[best]
            self.xF[i], self.xT[i] = 0.0, 0.0

    @staticmethod
    def _tri(off, di, rh):
        """Symmetric tridiagonal systems, one a row, by cyclic reduction: off[:, i]
        couples i and i + 1."""
        def sh(v, s, fill):
            o = torch.full_like(v, fill)
            if s > 0:
                o[:, s:] = v[:, :-s]
            else:
                o[:, :s] = v[:, -s:]
            return o
        a, c, b, d = sh(off, 1, 0.0), off.clone(), di, rh
        s = 1
        while s < di.shape[1]:
            al, ga = -a / sh(b, s, 1.0), -c / sh(b, -s, 1.0)
            b, d, a, c = (b + al * sh(c, s, 0.0) + ga * sh(a, -s, 0.0),
                          d + al * sh(d, s, 0.0) + ga * sh(d, -s, 0.0),
                          al * sh(a, s, 0.0), ga * sh(c, -s, 0.0))
            s *= 2
        return d / b

    def _integrate(self, mid):
        p = self.p
        if mid:
            i = torch.arange(self.ns, device=self.dev)
            o = _philox(i, i * 0, i * 0 + self.k // 2, i * 0, p.seed & 0xFFFFFFFF, p.seed >> 32)
            xi = torch.stack([(v.to(torch.float64) + 0.5) / 4294967296.0 - 0.5 for v in o[:3]], 1)
        new = self.r.clone()
        self.tension = torch.zeros(self.nb, dtype=torch.float64, device=self.dev)
        for g in self.groups:
            n, i, L, ok = g["n"], g["i"], g["L"], g["ok"]
            bond_ok = i < n - 1
            z1 = torch.zeros(len(n), 1, dtype=torch.float64, device=self.dev)
            z3 = torch.zeros(len(n), 1, 3, dtype=torch.float64, device=self.dev)
            prev = lambda v: torch.cat([z3 if v.dim() == 3 else z1, v[:, :-1]], 1)  # noqa: E731
            nxt = lambda v: torch.cat([v[:, 1:], z3 if v.dim() == 3 else z1], 1)  # noqa: E731
            B3, O3 = bond_ok[..., None], ok[..., None]
            u = self.u[g["bond"]]  # the last site holds the last bond's
            ub = u * B3
            um = prev(ub)
            in_cos = i < n - 2
            cos = _dot(u, nxt(u)) * in_cos
            t = u.clone()
            inner = (i > 0) & (i < n - 1)
            tt = um + u
            t = torch.where(inner[..., None], tt / tt.norm(dim=2, keepdim=True), u)
            gpar, gperp = g["gpar"], g["gperp"]
            one = torch.ones_like(cos)
            if mid:
                sp, sq = torch.sqrt(24.0 * gpar / p.delta), torch.sqrt(24.0 * gperp / p.delta)
                x = xi[g["site"]]
                fr = sq[..., None] * x + (sp - sq)[..., None] * t * _dot(t, x)[..., None]
                fr = fr * O3
                rh = _dot(nxt(fr) - fr, u) * bond_ok
                pt = self._tri(-cos, 2.0 * one, rh) * bond_ok
                fr = fr + pt[..., None] * ub - prev(pt)[..., None] * um
                self.fr[g["site"][ok]] = fr[ok]
            else:
                fr = self.fr[g["site"]] * O3
            half = 0.5 * self.F[g["bond"]] * B3
            tor = torch.cross(u, self.Tq[g["bond"]], dim=2) / g["bl"][..., None] * B3
            fs = prev(half) - prev(tor) + half + tor + fr
            # metric determinants
            dt, db = [one[:, 0], 2.0 * one[:, 0]], None
            c2 = cos * cos
            for j in range(2, L):
                dt.append(2.0 * dt[-1] - c2[:, j - 2] * dt[-2])
            dt = torch.stack(dt, 1)
            det = torch.gather(dt, 1, n - 1)
            # from the head: d[j] for site j, 1 at the last site, 2 before it
            bk = [None] * L
            last = n[:, 0] - 1
            cur, nx_ = one[:, 0], one[:, 0]
            for j in range(L - 1, -1, -1):
                v = 2.0 * cur - c2[:, j] * nx_
                v = torch.where(j >= last, one[:, 0],
                                torch.where(j == last - 1, 2.0 * one[:, 0], v))
                bk[j] = v
                cur, nx_ = v, cur
            bk = torch.stack(bk, 1)
            ahead = torch.cat([bk[:, 2:], one[:, :2]], 1)
            ke = (g["kappa"] + g["bl"] * cos * dt * ahead / det) / g["bl"] ** 2 * in_cos
            perp = lambda v, w: v - w * _dot(v, w)[..., None]  # noqa: E731
            up = nxt(u)
            umm, kem = prev(um), prev(ke)
            kemm = prev(kem)
            fs = fs + kemm[..., None] * perp(umm, um) \
                + kem[..., None] * (perp(u, um) - perp(um, u)) - ke[..., None] * perp(up, u)
            fs = fs * O3
            ip, dg = 1.0 / gperp, 1.0 / gpar - 1.0 / gperp
            mob = lambda v: ip[..., None] * v + dg[..., None] * t * _dot(t, v)[..., None]  # noqa: E731
            mf = mob(fs)
            tn = nxt(t)
            rh = _dot(nxt(mf) - mf, u) * bond_ok
            di = torch.where(bond_ok, 2.0 * ip + dg * (_dot(t, u) ** 2 + _dot(tn, u) ** 2), one)
            hu = (-ip * _dot(u, um) - dg * _dot(t, um) * _dot(t, u)) * (bond_ok & (i > 0))
            T = self._tri(nxt(hu), di, rh) * bond_ok
            self.tension[g["bond"][bond_ok]] = T[bond_ok]
            fs = fs + T[..., None] * ub - prev(T)[..., None] * um
            site = g["site"]
            start = self.r[site] if mid else self.rp[site]
            rn = start + (0.5 if mid else 1.0) * p.delta * mob(fs)
            o = (nxt(rn) - rn) * B3
            ln = o.norm(dim=2)
            bad = ((((g["bl"] - ln).abs() / g["bl"]) > 1e-3) & bond_ok).any(1)
            sw = self.switch[g["f"]] ^ bad
            self.switch[g["f"]] = sw
            st = g["bl"][..., None] * o / torch.where(bond_ok, ln, one)[..., None] * B3
            cum = prev(torch.cumsum(st, 1))
            head = torch.gather(rn, 1, (n - 1)[..., None].expand(-1, 1, 3))
            rest = torch.flip(torch.cumsum(torch.flip(st, [1]), 1), [1])
            fixed = torch.where(sw[:, None, None], rn[:, :1] + cum, head - rest)
            rn = torch.where(bad[:, None, None], fixed, rn)
            new[site[ok]] = rn[ok]
        if mid:
            self.rp = self.r.clone()
        self.r = new
        if not mid:
            d = self.r - self.dr0
            self.acc = self.acc + 2.0 * _dot(d, d)
            self.drmax = float(self.acc.max())
        self._bonds()

    def step(self, n, thermo=False):
        for _ in range(n):
            k = self.k + 1
            mid = k % 2 == 1
            if mid and k >= 3 and self.drmax > self.thr:
                self._rebuild()
            if self.nx and not mid:
                self._springs()
            self._pairs(thermo)
            if self.nx and not mid:
                # the partner search follows the pair pass of a full step
                self.k = k
                self._rebind()
                self.k = k - 1
            self._integrate(mid)
            self.k = k


def _soa(v):
    return v.T.contiguous().reshape(-1)


def exact(case, seed):
    if case["kind"] == "serve":
        return None  # minutes: hundreds of steps of every system
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p, fil = _system(case, seed)
    m = _Model(p, fil, dev)
    if case["kind"] == "analyse":
        off = torch.as_tensor(np.asarray(fil.site_off, dtype=np.int64), device=dev)
        n = off[1:] - off[:-1]
        fil_of = torch.repeat_interleave(torch.arange(fil.nf, device=dev), n)
        com = torch.zeros(fil.nf, 3, dtype=torch.float64, device=dev)
        com.index_add_(0, fil_of, m.r)
        com /= n[:, None]
        e2e = m.r[off[1:] - 1] - m.r[off[:-1]]
        return {"e2e": e2e.T.contiguous(), "com": com.T.contiguous(), "theta": None}
    if case["crosslinks"]:
        m.crosslinks(*_crosslinks(case, seed, p, fil))
    m.step(case["steps"], case["thermo"])
    out = {"r": _soa(m.r)}
    if case["precision"] == "fp64" and not case["crosslinks"]:
        out.update(r_prev=_soa(m.rp), f_rand=_soa(m.fr), force=_soa(m.F), torque=_soa(m.Tq),
                   tension=m.tension)
    if case["thermo"]:
        V = m.box ** 3
        pt = (m.nb * torch.eye(3, dtype=torch.float64, device=dev) + m.stress / case["steps"]) / V
        out.update(pressure_tensor=pt, pressure=float(pt.trace() / 3.0), volume=V, energy=m.E)
    return out
