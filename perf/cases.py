"""The measured cases: whole Poisson-Boltzmann calculations as users run them.

A case is one kind of call sequence on one problem:

  manual   driver.run_manual: one mg-manual input, objects made and freed in
           the call, potential mirrored to the host (the library's default)
  auto     driver.run_auto: an mg-auto focusing chain, the same way
  handle   a kept driver.Calc: fillco, solve, energy, the potential copied
           into a kept host buffer (a molecule rescored on one grid)
  forces   a kept Calc: fillco, solve, energy and the per-atom force
           components of the atoms a minimiser moves
  focus    a coarse solve giving the boundary of a large fine grid
  batch    several conformers filled, solved by driver.solve_batch
  served   binding triplets through the continuous-batching serve.Server

Grids run from 33^3 to 353^3, cubic and not; molecules from 12 to 60,000
atoms; lpbe and npbe; spline, molecular and smoothed surfaces; FP64, mixed and
mixed with the FP32-term boundary.  `exact` is the same discrete problem
solved to round-off in 64 bits with plain torch operations.
"""
import math

import numpy as np
import torch

from apbs_amd import driver, lib, serve, synth

SALT = [(1, 0.15, 2.0), (-1, 0.15, 2.0)]
SALT2 = [(1, 0.10, 2.0), (-1, 0.10, 2.0), (1, 0.05, 2.0), (-1, 0.05, 2.0)]


def listed():
    return [
        # the smallest calls: a small molecule on the smallest grid in use, where
        # latency, launches and object set-up are the cost
        dict(name="manual33_lpbe_smol_fp64", kind="manual", nx=33, ny=33, nz=33, atoms=12,
             h=0.45, npbe=False, srfm="smol", chgm="spl2", prec=0),
        # the usual input file of a small protein: two or three focusing levels
        dict(name="auto65_lpbe_smol_fp64", kind="auto", nx=65, ny=65, nz=65, atoms=900,
             h=0.0, npbe=False, srfm="smol", chgm="spl2", prec=0),
        # the 65^3 linear workload on a kept object
        dict(name="handle65_lpbe_spl2_fp64", kind="handle", nx=65, ny=65, nz=65, atoms=500,
             h=0.5, npbe=False, srfm="spl2", chgm="spl2", prec=0),
        # conformers of one ligand scored together, mixed precision
        dict(name="batch8_65_npbe_smol_mixed", kind="batch", nx=65, ny=65, nz=65, atoms=240,
             h=0.5, npbe=True, srfm="smol", chgm="spl2", prec=1, count=8),
        # solvation forces on a mid-sized solute
        dict(name="forces97_lpbe_spl2_fp64", kind="forces", nx=97, ny=97, nz=97, atoms=1500,
             h=0.0, npbe=False, srfm="spl2", chgm="spl2", prec=0),
        # a box that follows an elongated molecule: three different axes,
        # molecular surface, trilinear charges
        dict(name="ragged129x97x161_npbe_mol_fp64", kind="handle", nx=129, ny=97, nz=161,
             atoms=2400, h=0.0, npbe=True, srfm="mol", chgm="spl0", prec=0),
        # the 161^3 nonlinear workload, double precision and the fast mode
        dict(name="handle161_npbe_smol_fp64", kind="handle", nx=161, ny=161, nz=161, atoms=5000,
             h=0.4, npbe=True, srfm="smol", chgm="spl2", prec=0),
        dict(name="handle161_npbe_smol_fastbc", kind="handle", nx=161, ny=161, nz=161,
             atoms=5000, h=0.4, npbe=True, srfm="smol", chgm="spl2", prec=2),
        # a large linear solve in mixed precision
        dict(name="handle193_lpbe_spl2_mixed", kind="handle", nx=193, ny=193, nz=193,
             atoms=20000, h=0.35, npbe=False, srfm="spl2", chgm="spl2", prec=1),
        # four binding triplets of mixed sizes through the service
        dict(name="served12_triplets_fastbc", kind="served", nx=161, ny=161, nz=161, atoms=5000,
             h=0.0, npbe=True, srfm="smol", chgm="spl2", prec=2, count=12),
        # the largest: 97^3 coarse grid focused onto 353^3, 60,000 atoms
        dict(name="focus353_npbe_smol_mixed", kind="focus", nx=353, ny=353, nz=353, atoms=60000,
             h=0.3, npbe=True, srfm="smol", chgm="spl2", prec=1),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["manual", "auto", "handle", "handle", "handle", "forces", "batch",
                       "served"])
    npbe = rng.random() < 0.5
    srfm = rng.choice(["spl2", "smol", "mol"])
    chgm = rng.choice(["spl2", "spl2", "spl0"])
    prec = rng.choice([0, 1, 2])
    count = 1
    if kind == "manual":
        dims, npbe, prec = [rng.choice([33, 49, 65])] * 3, False, 0
        atoms = _logint(rng, 5, 120)
    elif kind == "auto":
        dims, npbe, chgm, prec = [rng.choice([65, 97])] * 3, False, "spl2", 0
        atoms = _logint(rng, 200, 2500)
    elif kind == "batch":
        dims, count = [rng.choice([49, 65, 97])] * 3, rng.choice([2, 3, 5, 8, 11])
        prec = rng.choice([0, 1])
        atoms = _logint(rng, 60, 900)
    elif kind == "forces":
        dims = [rng.choice([65, 97, 129]) for _ in range(3)]
        npbe, srfm, chgm, prec = False, "spl2", "spl2", 0
        atoms = _logint(rng, 200, 4000)
    elif kind == "served":
        dims, srfm, chgm, npbe = [161] * 3, "smol", "spl2", True
        count, atoms, prec = 3 * rng.choice([2, 3, 4]), _logint(rng, 600, 6000), rng.choice([1, 2])
    else:
        dims = [rng.choice([65, 97, 129, 161, 193, 225]) for _ in range(3)]
        if rng.random() < 0.5:
            dims = [dims[0]] * 3
        atoms = _logint(rng, 100, 12000)
    if npbe and srfm == "spl2":
        # salt in the gaps that narrow windows leave inside a large solute is a
        # badly conditioned problem that nobody poses
        srfm = "smol"
    return dict(kind=kind, nx=dims[0], ny=dims[1], nz=dims[2], atoms=atoms, h=0.0, npbe=npbe,
                srfm=srfm, chgm=chgm, prec=prec, count=count)


# ------------------------------------------------------------------ problems

def _pbe(case):
    return dict(npbe=case["npbe"], pdie=4.0 if case["npbe"] else 2.0, sdie=78.54,
                srfm=case["srfm"], chgm=case["chgm"], swin=0.3, srad=1.4, sdens=10.0,
                temp=298.15, bcfl="mdh", ions=SALT2 if case["atoms"] == 5000 else SALT)


def _axes(n, dims, h):
    """Semi-axes that hold n atoms at protein density, following the box (a box
    of given spacing holds them with at least 4 A to its faces)."""
    rad = (n / (math.sqrt(2.0) / 2.5 ** 3 * 0.9) * 3 / (4 * math.pi)) ** (1 / 3)
    rad = max(rad, 2.6)
    if h:
        half = 0.5 * h * (min(dims) - 1) - 4.0
        return (min(rad * 1.1, half),) * 2 + (min(rad, half),)
    m = float(np.prod(dims)) ** (1 / 3)
    return tuple(rad * (0.5 + 0.5 * d / m) for d in dims)


def _molecule(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    if case["atoms"] == 60000:
        axes = (50.0, 45.0, 40.0)
    elif case["atoms"] == 20000:
        axes = (30.0, 15.0, 15.0)
    elif case["atoms"] == 5000 and case["h"]:
        axes = (28.0, 24.0, 20.0)
    else:
        axes = _axes(case["atoms"], dims, case["h"])
    xyz, q, r, _ = synth.globule(case["atoms"], axes, seed, net_charge=-round(
        math.sqrt(case["atoms"]) / 7))
    return xyz, q, r


def _spacing(case, xyz, r):
    """The grid spacing: given, or the molecule's extent plus 7 A a side."""
    if case["h"]:
        return [case["h"]] * 3
    ext = xyz.max(0) - xyz.min(0) + 2 * (r.max() + 7.0)
    return [float(ext[d]) / (n - 1) for d, n in enumerate((case["nx"], case["ny"], case["nz"]))]


def _auto_lengths(xyz, r):
    ext = xyz.max(0) - xyz.min(0) + 2 * r.max()
    return [float(max(1.7 * v, 1.3 * (v + 20.0))) for v in ext], [float(v) for v in ext + 20.0]


def _conformers(case, seed):
    return [_molecule(dict(case, atoms=case["atoms"] + 7 * i), 1000 * seed + i)
            for i in range(case["count"])]


def _triplets(case, seed):
    """Binding triplets: a complex and the halves a random plane cuts it into,
    on one grid; the grids of a case are fixed, linear and nonlinear in turn."""
    rng = np.random.default_rng(seed)
    specs = []
    for t in range(case["count"] // 3):
        d = (161, 65, 129, 97)[t % 4]
        n = max(150, case["atoms"] >> (t % 4))
        xyz, q, r, _ = synth.globule(n, _axes(n, (d, d, d), 0.0), int(rng.integers(1 << 30)))
        side = (xyz - xyz.mean(0)) @ rng.normal(size=3) > 0
        grid = (xyz.max(0) - xyz.min(0) + 2 * (r.max() + 5.0)) / (d - 1)
        for sel in (np.ones(n, bool), side, ~side):
            specs.append(dict(xyz=xyz[sel], q=q[sel], r=r[sel], dime=(d, d, d), grid=grid,
                              center=0.5 * (xyz.min(0) + xyz.max(0)),
                              pbe=serve.LPBE if t % 2 else serve.NPBE))
    return specs


def _host(n):
    """A kept host buffer a potential is copied into."""
    return torch.empty(n, dtype=torch.float64, pin_memory=torch.cuda.is_available())


def _copy_potential(calc, buf):
    if not lib().Vpmg_copyArray(calc.pmg, 0, driver._dp(buf.numpy()), buf.numel()):
        raise RuntimeError("Vpmg_copyArray failed")
    return buf


def prepare(case, seed):
    pbe = _pbe(case)
    kind = case["kind"]
    dims = [case["nx"], case["ny"], case["nz"]]
    n = dims[0] * dims[1] * dims[2]
    st = dict(kind=kind, pbe=pbe, prec=case["prec"], dims=dims)
    if kind == "served":
        st["server"] = serve.Server(slots=8)
        st["requests"] = [serve.Request(s["xyz"], s["q"], s["r"], s["dime"], s["grid"],
                                        s["center"], s["pbe"], precision=case["prec"],
                                        want_potential=True, tag=i)
                          for i, s in enumerate(_triplets(case, seed))]
        return st
    if kind == "batch":
        st["mols"] = [driver.Molecule(*m) for m in _conformers(case, seed)]
        st["calcs"] = []
        for mol in st["mols"]:
            m = driver.manual_mgparm(dims, mol.center, grid=_spacing(case, mol.xyz, mol.r),
                                     chgm=pbe["chgm"])
            st["calcs"].append(driver.Calc(mol, m, pbe, precision=case["prec"], mirror=False))
        st["bufs"] = [_host(n) for _ in st["calcs"]]
        return st
    mol = driver.Molecule(*_molecule(case, seed))
    st["mol"] = mol
    st["grid"] = _spacing(case, mol.xyz, mol.r)
    if kind == "auto":
        st["cglen"], st["fglen"] = _auto_lengths(mol.xyz, mol.r)
    if kind in ("handle", "forces"):
        m = driver.manual_mgparm(dims, mol.center, grid=st["grid"], chgm=pbe["chgm"])
        st["calc"] = driver.Calc(mol, m, pbe, precision=case["prec"], mirror=False)
    if kind in ("handle", "forces", "focus"):
        st["buf"] = _host(n)
    if kind == "forces":
        st["movers"] = _movers(case)
    return st


def _movers(case):
    return list(range(0, case["atoms"], max(1, case["atoms"] // 32)))[:32]


def run(state):
    kind = state["kind"]
    if kind == "manual":
        e, calc = driver.run_manual(state["mol"], state["dims"], state["mol"].center,
                                    state["pbe"], grid=state["grid"])
        return e, calc.array("u")
    if kind == "auto":
        c = state["mol"].center
        energies, calc = driver.run_auto(state["mol"], state["dims"], state["cglen"],
                                         state["fglen"], c, c, state["pbe"])
        return np.array(energies), calc.array("u")
    if kind == "handle":
        calc = state["calc"]
        calc.fillco()
        calc.solve()
        return calc.energy(1), _copy_potential(calc, state["buf"])
    if kind == "forces":
        calc = state["calc"]
        calc.fillco()
        calc.solve()
        e = calc.energy(1)
        parts = [calc.force(a)[1:] for a in state["movers"]]
        qf, ib, db = (np.stack([p[k] for p in parts]) for k in range(3))
        return e, qf, ib, db, _copy_potential(calc, state["buf"])
    if kind == "batch":
        for calc in state["calcs"]:
            calc.fillco()
        if not all(driver.solve_batch(state["calcs"])):
            raise RuntimeError("a batched solve failed")
        energies = np.array([calc.energy(1) for calc in state["calcs"]])
        return energies, [_copy_potential(c, b) for c, b in zip(state["calcs"], state["bufs"])]
    if kind == "served":
        for req in state["requests"]:
            state["server"].submit(req)
        state["server"].drain()
        done = sorted(state["server"].poll(), key=lambda r: r["tag"])
        if any(r["status"] != 1 for r in done):
            raise RuntimeError("a served request failed")
        return (np.array([r["energy_kT"] for r in done]),
                [r.potential for r in state["requests"]])
    # focus: the coarse grid spans 1.2 A spacings, the fine one is given
    mol, pbe = state["mol"], state["pbe"]
    coarse = driver.Calc(mol, driver.manual_mgparm([97] * 3, mol.center, grid=[1.2] * 3), pbe,
                         mirror=False)
    coarse.fillco()
    coarse.solve()
    coarse.set_part_domain()
    fine = driver.Calc(mol, driver.manual_mgparm(state["dims"], mol.center, grid=state["grid"]),
                       pbe, old=coarse, precision=state["prec"], mirror=False)
    fine.fillco()
    fine.solve()
    fine.set_part_domain()
    return fine.energy(1), _copy_potential(fine, state["buf"])


def _grids(case):
    """(points, atoms, lpbe or npbe, 4 or 8 bytes in the cycles, calculations)."""
    n = case["nx"] * case["ny"] * case["nz"]
    word = 4 if case["prec"] else 8
    one = (n, case["atoms"], case["npbe"], word)
    if case["kind"] == "auto":
        return [one] * 3
    if case["kind"] == "focus":
        return [(97 ** 3, case["atoms"], True, 8), one]
    if case["kind"] == "batch":
        return [one] * case["count"]
    if case["kind"] == "served":
        return [((161, 65, 129, 97)[t % 4] ** 3, case["atoms"] >> (t % 4), t % 2 == 0, 4)
                for t in range(case["count"] // 3) for _ in range(3)]
    return [one]


def work(case):
    """Each solve reads the atoms, forms its five coefficient and charge maps
    once and writes the potential; each of its ten multigrid cycles (9 Newton
    steps of one cycle for npbe) reads the four operator arrays, the right-hand
    side and the solution once and writes the solution (13 operations a point
    and neighbour sum), the coarser levels a seventh of that again; npbe adds a
    residual with two exponentials a step in 64 bits."""
    by = fl = 0.0
    for n, atoms, npbe, word in _grids(case):
        by += 40.0 * atoms + 8.0 * n * (5 + 5 + 1)
        by += 10 * 7 * word * n * 8 / 7
        fl += 10 * 14.0 * n * 8 / 7
        if npbe:
            by += 10 * 8.0 * 7 * n
            fl += 10 * 60.0 * n
    return {"bytes": by, "flops": fl}


# --------------------------------------------------------------- 64-bit values

def _distance(a, b):
    return torch.sqrt(sum((a[:, None, d] - b[None, :, d]) ** 2 for d in range(3)))


class _Problem:
    """The discrete problem of one grid, solved to round-off in torch."""

    def __init__(self, atoms, dims, h, center, pbe, dev):
        self.dev, self.dims, self.h, self.pbe = dev, dims, [float(v) for v in h], pbe
        self.xyz, self.q, self.r = (self.t(v) for v in atoms)
        self.lo = [float(center[d]) - (dims[d] - 1) * self.h[d] / 2.0 for d in range(3)]
        self.hi = [float(center[d]) + (dims[d] - 1) * self.h[d] / 2.0 for d in range(3)]
        self.vol = self.h[0] * self.h[1] * self.h[2]
        na, ec, kb = 6.022045e23, 4.803242384e-10, 1.380662e-16
        ions = pbe["ions"]
        self.ionstr = sum(0.5 * c * q * q for q, c, _ in ions)
        self.irad = max(r for _, _, r in ions)
        self.xkappa = math.sqrt(self.ionstr * 1e-16 * (8.0 * math.pi * na * ec * ec) /
                                (1000.0 * pbe["sdie"] * kb * pbe["temp"]))
        self.zkappa2 = pbe["sdie"] * self.xkappa ** 2
        self.zmagic = 4.0 * math.pi * ec * ec / (kb * pbe["temp"]) * 1e8
        self.inside = self.inside_mask()
        self.fill_charge()
        self.spline() if pbe["srfm"] == "spl2" else self.molecular()

    def t(self, v):
        return torch.as_tensor(np.array(v, dtype=np.float64), device=self.dev)

    def inside_mask(self):
        ok = torch.ones(len(self.q), dtype=torch.bool, device=self.dev)
        for d in range(3):
            ok &= (self.xyz[:, d] > self.lo[d]) & (self.xyz[:, d] < self.hi[d])
        return ok

    def boxes(self, pos, reach, shift):
        """Indices and squared distances of the nodes around each centre: chunks
        of (centre numbers, flat index, distance^2, in range)."""
        nx, ny, nz = self.dims
        k = [int(math.ceil(reach / self.h[d])) + 1 for d in range(3)]
        off = [torch.arange(-k[d], k[d] + 2, device=self.dev) for d in range(3)]
        m = len(off[0]) * len(off[1]) * len(off[2])
        for c in torch.arange(len(pos), device=self.dev).split(max(1, 16000000 // m)):
            idx, d2, ok = [], [], []
            for d in range(3):
                p = pos[c, d] - self.lo[d] - shift[d] * self.h[d]
                i = torch.floor(p / self.h[d]).long()[:, None] + off[d][None]
                idx.append(i)
                d2.append((p[:, None] - self.h[d] * i.double()) ** 2)
                ok.append((i >= 0) & (i < self.dims[d]))
            flat = (idx[2][:, :, None, None] * ny + idx[1][:, None, :, None]) * nx + \
                idx[0][:, None, None, :]
            dd = d2[2][:, :, None, None] + d2[1][:, None, :, None] + d2[0][:, None, None, :]
            good = ok[2][:, :, None, None] & ok[1][:, None, :, None] & ok[0][:, None, None, :]
            yield c, flat, dd, good

    def marks(self, pos, rad, shift):
        out = torch.zeros(self.dims[0] * self.dims[1] * self.dims[2], dtype=torch.bool,
                          device=self.dev)
        if len(pos):
            for c, flat, dd, good in self.boxes(pos, float(rad.max()), shift):
                out[flat[good & (dd <= (rad[c] ** 2)[:, None, None, None])]] = True
        return out.reshape(self.dims[::-1])

    def windows(self, extra, shift):
        """The product over atoms of the cubic window in the distance."""
        w = self.pbe["swin"]
        ln = torch.zeros(self.dims[0] * self.dims[1] * self.dims[2], dtype=torch.float64,
                         device=self.dev)
        rad = self.r[self.inside] + extra
        for c, flat, dd, good in self.boxes(self.xyz[self.inside], float(rad.max()) + w, shift):
            a = rad[c][:, None, None, None]
            s = (torch.sqrt(dd) - a + w).clamp(0.0, 2 * w)
            v = 0.75 * s ** 2 / w ** 2 - 0.25 * s ** 3 / w ** 3
            ln.index_add_(0, flat[good], torch.log(v[good]))
        chi = torch.exp(ln)
        return torch.where(chi > 1e-12, chi, torch.zeros_like(chi)).reshape(self.dims[::-1])

    def spline(self):
        pd, sd = self.pbe["pdie"], self.pbe["sdie"]
        self.chi_eps = []
        for d in range(3):
            shift = [0.5 if e == d else 0.0 for e in range(3)]
            self.chi_eps.append(self.windows(0.0, shift))
        self.eps = [(sd - pd) * c + pd for c in self.chi_eps]
        self.kappa = self.windows(self.irad, [0.0] * 3)

    def sphere(self):
        srad = self.pbe["srad"]
        maxrad = float(self.r.max()) + max(self.irad, srad) + 0.5
        n = int(math.ceil(4.0 * math.pi * maxrad * maxrad * self.pbe["sdens"]))
        nth = int(math.floor(math.sqrt(math.pi * n / 4.0) + 0.5))
        pts = []
        for it in range(nth):
            th = math.pi / nth * it
            nph = int(math.floor(math.sin(th) * 2 * nth + 0.5))
            for ip in range(nph):
                ph = 2 * math.pi / nph * ip
                pts.append((math.cos(ph) * math.sin(th), math.sin(ph) * math.sin(th),
                            math.cos(th)))
        return self.t(pts)

    def accessible(self):
        """Points of the inflated atom spheres outside every other atom's."""
        ref, reach = self.sphere(), self.r + self.pbe["srad"]
        out, num = [], torch.arange(len(self.q), device=self.dev)
        for c in num.split(64):
            d = _distance(self.xyz[c], self.xyz)
            near = (d < reach[c][:, None] + reach[None] + 1e-6) & (c[:, None] != num[None])
            cnt = int(near.sum(1).max())
            nb = torch.argsort((~near).to(torch.int8), dim=1, stable=True)[:, :max(cnt, 1)]
            use = torch.gather(near, 1, nb)
            pts = reach[c][:, None, None] * ref[None] + self.xyz[c][:, None]
            free = torch.ones(pts.shape[:2], dtype=torch.bool, device=self.dev)
            for k in range(nb.shape[1]):
                d2 = ((pts - self.xyz[nb[:, k]][:, None]) ** 2).sum(-1)
                free &= ~((d2 < (reach[nb[:, k]] ** 2)[:, None]) & use[:, k][:, None])
            out.append(pts[free])
        return torch.cat(out)

    def molecular(self):
        pd, sd = self.pbe["pdie"], self.pbe["sdie"]
        sas = self.accessible()
        srad = torch.full((len(sas),), self.pbe["srad"], dtype=torch.float64, device=self.dev)
        inv = []
        for d in range(3):
            shift = [0.5 if e == d else 0.0 for e in range(3)]
            solute = self.marks(self.xyz[self.inside], self.r[self.inside] + self.pbe["srad"],
                                shift)
            solute &= ~self.marks(sas, srad, shift)
            s = solute.double()
            inv.append(s / pd + (1.0 - s) / sd)
        self.kappa = (~self.marks(self.xyz, self.r + self.irad, [0.0] * 3)).to(torch.float64)
        self.eps = [1.0 / v for v in inv]
        if self.pbe["srfm"] == "smol":
            self.eps = [self.harmonic(inv, d) for d in range(3)]

    def harmonic(self, inv, d):
        """The harmonic mean of a face's value and its eight neighbours'."""
        tot, num = inv[d].clone(), torch.ones_like(inv[d])
        for e in range(3):
            if e == d:
                continue
            for sd, se in ((0, 0), (0, -1), (1, 0), (1, -1)):
                v = [0, 0, 0]
                v[2 - d], v[2 - e] = sd, se
                dst = tuple(slice(max(0, -s), n - max(0, s)) for s, n in zip(v, tot.shape))
                src = tuple(slice(max(0, s), n - max(0, -s)) for s, n in zip(v, tot.shape))
                tot[dst] += inv[e][src]
                num[dst] += 1.0
        return num / tot

    def fill_charge(self):
        nx, ny, _ = self.dims
        self.charge = torch.zeros(nx * ny * self.dims[2], dtype=torch.float64, device=self.dev)
        width = 2 if self.pbe["chgm"] == "spl2" else 1
        lists = []
        for d in range(3):
            f = (self.xyz[:, d] - self.lo[d]) / self.h[d]
            i = torch.floor(f).long()[:, None] + torch.arange(1 - width, width + 1,
                                                              device=self.dev)[None]
            x = i - f[:, None]
            if width == 2:
                v = torch.where(x.abs() <= 0.5, 0.75 - x * x, 0.5 * (1.5 - x.abs()).clamp(min=0) ** 2)
            else:
                v = (1.0 - x.abs()).clamp(min=0.0)
            lists.append((i, v))
        (i, wx), (j, wy), (k, wz) = lists
        flat = (k[:, :, None, None] * ny + j[:, None, :, None]) * nx + i[:, None, None, :]
        w = wz[:, :, None, None] * wy[:, None, :, None] * wx[:, None, None, :]
        self.weights, self.nodes = w.reshape(len(self.q), -1), flat.reshape(len(self.q), -1)
        self.charge.index_add_(0, self.nodes.reshape(-1), (
            self.weights * (self.q * self.zmagic / self.vol)[:, None]).reshape(-1))
        self.charge = self.charge.reshape(self.dims[::-1])

    def shell(self):
        m = torch.ones(self.dims[::-1], dtype=torch.bool, device=self.dev)
        m[1:-1, 1:-1, 1:-1] = False
        k, j, i = (v.double() for v in torch.nonzero(m, as_tuple=True))
        at = torch.stack([self.lo[0] + self.h[0] * i, self.lo[1] + self.h[1] * j,
                          self.lo[2] + self.h[2] * k], 1)
        return m, at

    def mdh(self):
        ec, kb, eps0 = 1.6021773e-19, 1.3806581e-23, 8.8541878e-12
        pre = ec / (4 * math.pi * eps0 * self.pbe["sdie"] * kb * self.pbe["temp"]) * 1e10
        m, at = self.shell()
        fac = pre * ec * self.q / (1 + self.xkappa * self.r)
        val = []
        for c in at.split(max(1, 20000000 // len(self.q))):
            d = _distance(c, self.xyz)
            val.append((fac[None] * torch.exp(-self.xkappa * (d - self.r[None])) / d).sum(1))
        u = torch.zeros(self.dims[::-1], dtype=torch.float64, device=self.dev)
        u[m] = torch.cat(val)
        return u

    def focused(self, old):
        """Boundary values interpolated in the solution of a coarser problem."""
        m, at = self.shell()
        w = torch.zeros(len(at), dtype=torch.float64, device=self.dev)
        f = [((at[:, d] - old.lo[d]) / old.h[d]).clamp(0.0, old.dims[d] - 1.0) for d in range(3)]
        b = [torch.floor(v).long().clamp(max=n - 2) for v, n in zip(f, old.dims)]
        for c in range(8):
            o = [(c >> d) & 1 for d in range(3)]
            t = torch.ones_like(w)
            for d in range(3):
                s = f[d] - b[d]
                t = t * (s if o[d] else 1.0 - s)
            w += t * old.u[b[2] + o[2], b[1] + o[1], b[0] + o[0]]
        u = torch.zeros(self.dims[::-1], dtype=torch.float64, device=self.dev)
        u[m] = w
        return u

    def apply(self, u):
        """Sum over faces of c eps (u - neighbour) at the interior nodes."""
        out = torch.zeros_like(u)
        mid = slice(1, -1)
        for d in range(3):
            c = self.vol / self.h[d] ** 2
            ax = 2 - d
            flux = c * torch.diff(u, dim=ax) * self.eps[d].narrow(ax, 0, u.shape[ax] - 1)
            out[mid, mid, mid] -= torch.diff(flux, dim=ax)[
                tuple(slice(None) if e == ax else mid for e in range(3))]
        return out

    def diagonal(self):
        out = torch.ones_like(self.kappa)
        mid = slice(1, -1)
        tot = 0
        for d in range(3):
            c, e = self.vol / self.h[d] ** 2, self.eps[d]
            lo = [mid] * 3
            lo[2 - d] = slice(0, -2)
            tot = tot + c * (e[mid, mid, mid] + e[tuple(lo)])
        out[mid, mid, mid] = tot
        return out

    def cg(self, extra, b, tol):
        """(A + extra) x = b by conjugate gradients with the diagonal."""
        inner = torch.zeros_like(b)
        inner[1:-1, 1:-1, 1:-1] = 1.0
        minv = inner / (self.diag + extra)
        extra = extra * inner
        x, r = torch.zeros_like(b), b * inner
        z = minv * r
        p, rz = z.clone(), (r * z).sum()
        stop = tol * tol * rz
        for it in range(6000):
            ap = self.apply(p) + extra * p
            a = rz / (p * ap).sum()
            x += a * p
            r -= a * ap
            z = minv * r
            new = (r * z).sum()
            if it % 16 == 15 and float(new) <= float(stop):
                break
            p = z + (new / rz) * p
            rz = new
        return x

    def solve(self, u):
        self.diag = self.diagonal()
        ck = self.vol * self.zkappa2 * self.kappa
        f = self.vol * self.charge
        mid = (slice(1, -1),) * 3
        if not self.pbe.get("npbe"):
            self.u = u + self.cg(ck, f - self.apply(u), 1e-13)
            return self
        terms = [(0.5 / self.ionstr * c, q) for q, c, _ in self.pbe["ions"]]

        def residual(v):
            out = f - self.apply(v)
            for s, q in terms:
                out += s * q * ck * torch.exp((-q * v).clamp(-85.0, 85.0))
            keep = torch.zeros_like(out)
            keep[mid] = out[mid]
            return keep

        r = residual(u)
        first = norm = float(r.abs().sum())
        for _ in range(40):
            jac = sum(s * q * q * ck * torch.exp((-q * u).clamp(-85.0, 85.0)) for s, q in terms)
            du = self.cg(jac, r, 1e-10)
            step = 1.0
            while True:
                rt = residual(u + step * du)
                nt = float(rt.abs().sum())
                if nt < norm or step < 1e-3 or norm < 1e-12 * first:
                    break
                step *= 0.5
            u, r, norm = u + step * du, rt, nt
            if norm < 1e-12 * first:
                break
        self.u = u
        return self

    def energy(self):
        if self.pbe["chgm"] == "spl2":
            qf = float((self.u * self.charge).sum()) * self.vol / self.zmagic
        else:
            qf = float((self.u.reshape(-1)[self.nodes] * self.weights * self.q[:, None]).sum())
        if not self.pbe.get("npbe"):
            return 0.5 * qf
        low = tuple(slice(0, n - 1) for n in self.u.shape)
        di = sum(float((self.eps[d][low] * (torch.diff(self.u, dim=2 - d)[low] /
                                            self.h[d]) ** 2).sum()) for d in range(3))
        di = 0.5 * di * self.vol / self.zmagic
        qm = 0.0
        for q, c, _ in self.pbe["ions"]:
            salt = torch.where(self.kappa > 0, self.u, torch.zeros_like(self.u))
            qm += float((self.kappa * c * (torch.exp(-q * salt) - 1.0)).sum())
        qm *= 0.5 * self.zkappa2 / self.ionstr * self.vol / self.zmagic
        return qf - di - qm

    def forces(self, atoms):
        """The three force components of a linear problem with spline windows."""
        qf, ib, db = (np.zeros((len(atoms), 3)) for _ in range(3))
        w, deps = self.pbe["swin"], self.pbe["sdie"] - self.pbe["pdie"]
        h = self.t(self.h)

        def slope(at, pos, rad):
            """-(window'/window) times the unit vector from the atom."""
            v = at - pos
            d = torch.sqrt((v * v).sum(-1))
            s = d - rad + w
            ok = (s > 1e-9) & (s < 2 * w - 1e-9)
            s = torch.where(ok, s, torch.full_like(s, w))
            g = (1.5 * s / w ** 2 - 0.75 * s * s / w ** 3) / (
                0.75 * s * s / w ** 2 - 0.25 * s ** 3 / w ** 3)
            return torch.where(ok, -g / d, torch.zeros_like(g))[..., None] * v

        for n, a in enumerate(atoms):
            pos, rad = self.xyz[a], self.r[a]
            # fixed charges: the derivative of the quadratic B-spline weights
            val, der, sl = [], [], []
            for d in range(3):
                f = float((pos[d] - self.lo[d]) / self.h[d])
                i = torch.arange(int(math.floor(f)) - 1, int(math.floor(f)) + 3,
                                 dtype=torch.float64, device=self.dev)
                x = i - f
                val.append(torch.where(x.abs() <= 0.5, 0.75 - x * x,
                                       0.5 * (1.5 - x.abs()).clamp(min=0) ** 2))
                der.append(torch.where(x.abs() <= 0.5, -2.0 * x,
                                       -torch.sign(x) * (1.5 - x.abs()).clamp(min=0)))
                sl.append(slice(int(i[0]), int(i[-1]) + 1))
            box = self.u[sl[2], sl[1], sl[0]]
            for d in range(3):
                v = [der[e] if e == d else val[e] for e in range(3)]
                qf[n, d] = float(self.q[a] / self.h[d] * torch.einsum(
                    "kji,k,j,i->", box, v[2], v[1], v[0]))
            # the nodes around the atom, with one more for the differences
            reach = float(rad) + self.irad + w + max(self.h)
            lo = [int(math.floor((float(pos[d]) - self.lo[d] - reach) / self.h[d])) - 1
                  for d in range(3)]
            hi = [int(math.ceil((float(pos[d]) - self.lo[d] + reach) / self.h[d])) + 2
                  for d in range(3)]
            g = [torch.arange(lo[d], hi[d], device=self.dev, dtype=torch.float64) for d in range(3)]
            at = torch.stack(torch.meshgrid(g[2], g[1], g[0], indexing="ij")[::-1], -1) * h + \
                self.t(self.lo)
            cut = tuple(slice(lo[d], hi[d]) for d in (2, 1, 0))
            u, kap = self.u[cut], self.kappa[cut]
            tg = slope(at, pos, rad + self.irad)
            keep = ((at - pos) ** 2).sum(-1) <= (rad + self.irad + w) ** 2
            ib[n] = ((keep * u * u * kap)[..., None] * tg).sum((0, 1, 2)).cpu().numpy() * (
                0.5 * self.zkappa2 * self.vol / self.zmagic)
            rtot = float(rad) + w + w
            if any(float(pos[d]) <= self.lo[d] + rtot or float(pos[d]) >= self.hi[d] - rtot
                   for d in range(3)):
                continue
            tot = torch.zeros(3, dtype=torch.float64, device=self.dev)
            for d in range(3):
                half = torch.zeros(3, dtype=torch.float64, device=self.dev)
                half[d] = 0.5 * self.h[d]
                dh = slope(at + half, pos, rad) * self.chi_eps[d][cut][..., None]
                du = torch.diff(u, dim=2 - d)
                ax, m = 2 - d, u.shape[2 - d]
                # a face adds u_low * du from its lower node and -u_high * du from its upper
                tot += ((-(du * du)[..., None] * dh.narrow(ax, 0, m - 1)) /
                        self.h[d] ** 2).sum((0, 1, 2))
            db[n] = (-tot * self.vol * deps * 0.5 / self.zmagic).cpu().numpy()
        return qf, ib, db


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    n = case["nx"] * case["ny"] * case["nz"] * case.get("count", 1)
    if case["kind"] == "focus" or (dev.type == "cpu" and n > 400000):
        return None                   # minutes of conjugate gradients
    pbe = _pbe(case)
    dims = [case["nx"], case["ny"], case["nz"]]

    def solved(atoms, dims, h, center, pbe):
        p = _Problem(atoms, dims, h, center, pbe, dev)
        return p.solve(p.mdh())

    def mid(xyz):
        return 0.5 * (xyz.max(0) + xyz.min(0))

    if case["kind"] == "served":
        done = [solved((s["xyz"], s["q"], s["r"]), list(s["dime"]), s["grid"], s["center"],
                       s["pbe"]) for s in _triplets(case, seed)]
        return np.array([p.energy() for p in done]), [p.u.reshape(-1).cpu().numpy() for p in done]
    if case["kind"] == "batch":
        done = [solved(a, dims, _spacing(case, a[0], a[2]), mid(a[0]), pbe)
                for a in _conformers(case, seed)]
        return np.array([p.energy() for p in done]), [p.u.reshape(-1).cpu() for p in done]
    atoms = _molecule(case, seed)
    c = mid(atoms[0])
    kJ = driver.kT_to_kJmol(1.0, pbe["temp"])
    if case["kind"] == "auto":
        cglen, fglen = _auto_lengths(atoms[0], atoms[2])
        grids = _focus_grids(dims, cglen, fglen)
        energies, prev = [], None
        for h in grids:
            p = _Problem(atoms, dims, h, c, pbe, dev)
            prev = p.solve(p.mdh() if prev is None else p.focused(prev))
            energies.append(kJ * p.energy())
        return np.array(energies), prev.u.cpu().numpy()
    p = solved(atoms, dims, _spacing(case, atoms[0], atoms[2]), c, pbe)
    if case["kind"] == "manual":
        return kJ * p.energy(), p.u.cpu().numpy()
    if case["kind"] == "forces":
        return (p.energy(), *p.forces(_movers(case)), p.u.reshape(-1).cpu())
    return p.energy(), p.u.reshape(-1).cpu()


def _focus_grids(dims, cglen, fglen):
    """Spacings of an mg-auto chain: a constant ratio a level, at most four-fold."""
    cg = [cglen[d] / (dims[d] - 1) for d in range(3)]
    fg = [fglen[d] / (dims[d] - 1) for d in range(3)]
    levels = max(2 if f / c >= 0.25 else int(math.ceil(math.log(f / c) / math.log(0.25))) + 1
                 for c, f in zip(cg, fg))
    ratio = [(f / c) ** (1.0 / (levels - 1.0)) for c, f in zip(cg, fg)]
    return [[c * r ** k for c, r in zip(cg, ratio)] for k in range(levels)]
