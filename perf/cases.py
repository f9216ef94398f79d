"""The work a program gives this framework, as cases that can be timed and compared.

Every case goes through the MDLIB-named calls of `msmpscu_amd.mdlib` (and `DeviceForceMatch` of
`msmpscu_amd.adjoint`), on host arrays in and out, in eV, Angstrom and fs.  Kinds:

  md      a segment of molecular dynamics of one or many boxes: For_One_Steps, then the state
          copied out; the state goes on from pass to pass, as a trajectory does
  eval    a new configuration in an existing context: positions in, list, forces, energies out
  quench  damped dynamics of a set of images from given positions
  fit     loss and coefficient gradient of force matching on a set of boxes
  stress  per-atom stress and virial of a stored configuration

`draw` gives more cases of the same kinds over the same ranges: boxes of 250 to a million atoms,
one or two species, FS and EAM tables of 2000 to 10000 knots, 100 K to 1200 K, bulk and films.
"""
import math

import numpy as np

from msmpscu_amd import adjoint as adj
from msmpscu_amd import configs as cfg
from msmpscu_amd import mdlib as md

KB = 8.617333262e-5      # eV / K, for the initial velocities
W_A, W_RC = 3.165, 4.4002
CUNI_A, CUNI_RC = 3.57, 6.0
SKIN = 0.3


# ------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------

def _w(kind, cells, **kw):
    c = {"kind": kind, "alloy": False, "nx": cells[0], "ny": cells[1], "nz": cells[2],
         "nbox": 1, "spread": 1.0, "pot": "FS_TYPE", "ntab": 5000, "mx": 64, "temp": 300.0,
         "vac": 0.0, "film": False, "steps": 1}
    c.update(kw)
    return c


def _cuni(cells, **kw):
    d = {"alloy": True, "temp": 1200.0, "film": True, "mx": 160}
    d.update(kw)
    return _w("md", cells, **d)


def listed():
    return [
        # a box of point-defect studies: two thousand atoms, where launches and latency count
        _w("md", (10, 10, 10), name="md_w_2k", steps=200, vac=0.002),
        # an ordinary box with a tabulated embedding function
        _w("md", (20, 20, 20), name="md_w_16k_eam", steps=100, pot="EAM_TYPE", temp=600.0),
        # a box of odd sides, hot, one per cent of its sites empty
        _w("md", (39, 41, 43), name="md_w_137k", steps=100, temp=900.0, vac=0.01),
        # the largest plain box (the benchmark's): a million atoms, list capacity 32
        _w("md", (80, 80, 80), name="md_w_1m", steps=500, vac=0.005, mx=32),
        # a small alloy film: two species, three table kinds, eighty neighbours an atom
        _cuni((10, 11, 9), name="md_cuni_4k", steps=100),
        # a large alloy film
        _cuni((48, 47, 49), name="md_cuni_442k", steps=50),
        # many uneven boxes advanced together (replicas)
        _w("md", (14, 14, 14), name="md_batch_64", nbox=64, spread=3.0, steps=100, temp=700.0,
           vac=0.001),
        # one image of a path or a trial configuration: positions in, forces and energies out
        _w("eval", (8, 8, 8), name="eval_w_1k"),
        # the same for an ordinary box, tabulated embedding
        _w("eval", (30, 30, 30), name="eval_w_54k_eam", pot="EAM_TYPE", vac=0.002),
        # a string of sixteen images relaxed by damped dynamics
        _w("quench", (8, 8, 8), name="quench_16x1k", nbox=16, steps=50, vac=0.002),
        # one gradient of a potential fit (the benchmark's set of boxes)
        _w("fit", (8, 8, 8), name="fit_64x1k_eam", nbox=64, pot="EAM_TYPE"),
        # analysis of a stored snapshot
        _w("stress", (30, 31, 29), name="stress_w_54k", temp=900.0, vac=0.002),
    ]


def _loguni(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _sides(rng, sites, per_cell, least):
    c = (sites / per_cell) ** (1.0 / 3.0)
    return tuple(max(least, int(round(c * rng.uniform(0.85, 1.18)))) for _ in range(3))


def draw(rng):
    kind = rng.choice(["md", "md", "md", "alloy", "alloy", "batch", "batch", "eval", "eval",
                       "quench", "fit", "stress"])
    common = {"pot": rng.choice(["FS_TYPE", "EAM_TYPE"]),
              "ntab": rng.choice([2000, 5000, 5000, 5000, 10000]),
              "temp": round(rng.uniform(100.0, 1200.0), 1),
              "vac": rng.choice([0.0, 0.001, 0.005, 0.01])}
    if kind == "md":
        n = _loguni(rng, 250, 1.0e6)
        return _w("md", _sides(rng, n, 2, 5), steps=int(min(200, max(20, 5.0e7 / n))),
                  film=rng.random() < 0.2, **common)
    if kind == "alloy":
        n = _loguni(rng, 900, 4.0e5)
        return _cuni(_sides(rng, n, 4, 6), steps=int(min(100, max(15, 1.5e7 / n))),
                     film=rng.random() < 0.6, **common)
    if kind == "batch":
        nbox = int(round(_loguni(rng, 4, 128)))
        n = _loguni(rng, 500, min(16000.0, 8.0e5 / nbox))
        return _w("md", _sides(rng, n, 2, 6), nbox=nbox, spread=round(rng.uniform(1.0, 4.0), 2),
                  steps=int(min(100, max(20, 4.0e7 / (n * nbox)))), **common)
    if kind == "eval":
        return _w("eval", _sides(rng, _loguni(rng, 250, 2.0e5), 2, 5), **common)
    if kind == "quench":
        nbox = rng.randint(1, 24)
        return _w("quench", _sides(rng, _loguni(rng, 400, 6000), 2, 6), nbox=nbox,
                  steps=rng.randint(20, 60), **common)
    if kind == "fit":
        common["vac"] = 0.0
        return _w("fit", _sides(rng, _loguni(rng, 250, 1500), 2, 5), nbox=rng.randint(4, 64),
                  **common)
    return _w("stress", _sides(rng, _loguni(rng, 1000, 1.0e5), 2, 6), **common)


# ------------------------------------------------------------------------------------------
# inputs, from the seed alone
# ------------------------------------------------------------------------------------------

def _box_sides(case):
    """Cells of every box; spread s: sides between 1/cbrt(s) and cbrt(s) times the mean."""
    sides, nb = (case["nx"], case["ny"], case["nz"]), case["nbox"]
    if nb == 1 or case["spread"] == 1.0:
        return [sides] * nb
    out = []
    for k in range(nb):
        f = case["spread"] ** ((2.0 * ((k * 29) % nb) / (nb - 1) - 1.0) / 3.0)
        out.append(tuple(max(5, int(round(c * f))) for c in sides))
    return out


def _one_box(case, sides, rng):
    """dict of numpy arrays: x, v (n, 3), ityp (0-based), mass per group, lo, ln, ifpd."""
    a = CUNI_A if case["alloy"] else W_A
    basis = (np.array([[0, 0, 0], [.5, .5, 0], [.5, 0, .5], [0, .5, .5]]) if case["alloy"] else
             np.array([[0, 0, 0], [.5, .5, .5]]))
    g = np.stack(np.meshgrid(*(np.arange(s) for s in sides), indexing="ij"), -1).reshape(-1, 3)
    x = ((g[:, None, :] + basis[None]).reshape(-1, 3) + 0.25) * a
    ln = np.array(sides) * a
    if case["vac"] > 0:
        keep = np.ones(len(x), bool)
        keep[rng.choice(len(x), max(1, int(round(case["vac"] * len(x)))), replace=False)] = False
        x = x[keep]
    x = x - 0.5 * ln
    ifpd = (1, 1, 1)
    if case["film"]:
        ln = ln + np.array([0.0, 0.0, 40.0])
        ifpd = (1, 1, 0)
    if case["kind"] == "fit":   # boxes of a fit differ by a small homogeneous strain
        f = 1.0 + rng.uniform(-0.02, 0.02, 3)
        x, ln = x * f, ln * f
    n = len(x)
    x = x + rng.normal(0.0, 0.1 if case["kind"] == "fit" else 0.05, x.shape)
    lo = -0.5 * ln
    for k in range(3):
        if ifpd[k]:
            x[:, k] = np.where(x[:, k] < lo[k], x[:, k] + ln[k],
                               np.where(x[:, k] >= lo[k] + ln[k], x[:, k] - ln[k], x[:, k]))
    if case["alloy"]:
        ityp = (rng.permutation(n) < n // 2).astype(np.int32)
        order = np.argsort(ityp, kind="stable")   # atoms grouped by species
        x, ityp = x[order], ityp[order]
        mass = np.array([cfg.CU_MASS, cfg.NI_MASS]) * cfg.AMU
    else:
        ityp, mass = np.zeros(n, np.int32), np.array([cfg.W_MASS]) * cfg.AMU
    if case["kind"] == "md":
        m = mass[ityp][:, None]
        v = rng.normal(0.0, 1.0, x.shape) * np.sqrt(KB * case["temp"] / m)
        v -= (m * v).sum(0) / m.sum()
    else:
        v = np.zeros_like(x)
    return {"x": x, "v": v, "ityp": ityp, "mass": mass, "lo": lo, "ln": ln, "ifpd": ifpd}


def _inputs(case, seed):
    rng = np.random.default_rng([seed, 20])
    return [_one_box(case, s, rng) for s in _box_sides(case)]


def _ctrl(case):
    ntab = case["ntab"]
    if case["alloy"]:
        c = cfg.cuni_ctrl(mx=case["mx"], ntab=ntab)
        c.NUMFTABE = ntab
    else:
        c = cfg.w_ctrl(mx=case["mx"], ntab=ntab, nembd=ntab)
    c.IFPD = (1, 1, 0) if case["film"] else (1, 1, 1)
    return c


def _simbox(case, b):
    g = len(b["mass"])
    pt = np.array([[1, 3], [3, 2]] if g == 2 else [[1]], dtype=np.int32)
    return md.SimMDBox(NPRT=len(b["x"]), NGROUP=g, ZL=b["ln"], BOXLOW=b["lo"], XP=b["x"],
                       XP1=b["v"], ITYP=b["ityp"] + 1, STATU=np.ones(len(b["x"]), np.int32),
                       CM=b["mass"], PTYPE=pt, SYMB=["Cu", "Ni"] if g == 2 else ["W"],
                       RR=CUNI_A if g == 2 else W_A)


def _thomas(v):
    """c with (c[i-1] + 4 c[i] + c[i+1]) / 6 = v[i] (c zero outside)."""
    n = len(v)
    w, c = np.empty(n), np.empty(n)
    w[0], c[0] = 0.25, v[0] * 6.0 / 4.0
    for i in range(1, n):
        d = 4.0 - w[i - 1]
        w[i], c[i] = 1.0 / d, (6.0 * v[i] - c[i - 1]) / d
    for i in range(n - 2, -1, -1):
        c[i] -= w[i] * c[i + 1]
    return c


def _coefficients(case, seed):
    """Spline coefficients of the trial potential and of the one the targets come from."""
    t = _tables(case)
    n = case["ntab"]
    r = (np.arange(1, n + 1) / t["csi"]) ** 2
    c = np.zeros((3, n))
    c[0], c[1] = _thomas(t["potr"][0, 1:n + 1] / r), _thomas(t["potb"][0, 1:n + 1])
    if case["pot"] == "EAM_TYPE":
        c[2] = _thomas(t["femb"][1:n + 1])
    rng = np.random.default_rng([seed, 21])
    return c, c * (1.0 + 0.01 * rng.normal(size=c.shape))


def prepare(case, seed):
    raw = _inputs(case, seed)
    boxes = [_simbox(case, b) for b in raw]
    ctrl = _ctrl(case)
    ft = (cfg.cuni_forcetable if case["alloy"] else cfg.w_forcetable)(boxes[0], ctrl,
                                                                      case["pot"])
    if case["kind"] == "fit":
        fm = adj.DeviceForceMatch(boxes, ctrl, ft)
        c, target = _coefficients(case, seed)
        fm.set_targets(target)
        return {"kind": "fit", "fm": fm, "c": c}
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(case["pot"], fc)
    md.Initialize_Globle_Variables_DEV(boxes, ctrl, fc)
    md.Init_Forcetable_Dev(boxes, ctrl, fc)
    md.Cal_NeighBoreList_DEV(boxes, ctrl, fc)
    md.CalForce_ForceClass(boxes, ctrl, fc)
    s = {"kind": case["kind"], "boxes": boxes, "ctrl": ctrl, "fc": fc, "steps": case["steps"],
         "time": 0}
    if case["kind"] in ("eval", "quench"):
        # the configuration the pass brings in: every atom moved a little
        rng = np.random.default_rng([seed, 22])
        x = np.concatenate([b["x"] for b in raw])
        lo = np.concatenate([np.tile(b["lo"], (len(b["x"]), 1)) for b in raw])
        ln = np.concatenate([np.tile(b["ln"], (len(b["x"]), 1)) for b in raw])
        x = x + rng.normal(0.0, 0.03, x.shape)
        per = np.array(raw[0]["ifpd"], bool)
        x = np.where(per & (x < lo), x + ln, np.where(per & (x >= lo + ln), x - ln, x))
        s["x"], s["v"] = x, np.zeros_like(x)
    return s


# ------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------

def run(s):
    if s["kind"] == "fit":
        loss, grad = s["fm"].loss_and_grad(s["c"])
        return {"loss": loss, "grad": grad}
    boxes, ctrl, fc = s["boxes"], s["ctrl"], s["fc"]
    dev = fc.Device
    if s["kind"] == "md":
        md.For_One_Steps(s["time"], s["steps"], boxes, ctrl, fc)
        s["time"] += s["steps"]
        x, v, f, st, dis = dev.get_atoms()
        return {"x": x, "v": v, "f": f, "statu": st, "dis": dis}
    if s["kind"] == "eval":
        dev.put_atoms(s["x"])
        md.Cal_NeighBoreList_DEV(boxes, ctrl, fc)
        md.CalForce_ForceClass(boxes, ctrl, fc)
        md.CalEpot_ForceClass(boxes, ctrl, fc)
        return {"f": dev.get_forces(), "epot": dev.get_epot(), "e": dev.get_box_epot()}
    if s["kind"] == "quench":
        dev.put_atoms(s["x"], s["v"])
        md.Cal_NeighBoreList_DEV(boxes, ctrl, fc)
        md.CalForce_ForceClass(boxes, ctrl, fc)
        dev.dyn_damp(s["steps"], 1.0e-10, ctrl.H)
        x, v, f, st, dis = dev.get_atoms()
        return {"x": x, "v": v, "f": f, "epot": dev.get_epot(), "e": dev.get_box_epot()}
    return {"avp": md.Cal_AtomicStress(boxes, ctrl, fc),
            "vir": md.CalPTensor_ForceClass(boxes, ctrl, fc), "f": dev.get_forces()}


def _atoms(case):
    per = 4 if case["alloy"] else 2
    n = sum(a * b * c for a, b, c in _box_sides(case)) * per
    return n * (1.0 - case["vac"])


def work(case):
    """Bytes and operations a pass cannot do without, with the mean list length K: a step reads
    and writes positions, velocities and displacements once, reads the list in both passes and
    writes and reads F'; a pair costs about 25 operations for the density and 40 for the force."""
    n, k = _atoms(case), 86.0 if case["alloy"] else 26.0
    lst, pair = 4.0 * k + 4.0, 65.0 * k
    out = n * (12 * 8 + 4)
    if case["kind"] == "md":
        every = 5 if case["alloy"] else 10
        step = n * (144.0 + 2 * lst + 16.0) + n * (lst + 24.0) / every
        return {"bytes": step * case["steps"] + out, "flops": n * pair * case["steps"]}
    if case["kind"] == "eval":
        return {"bytes": n * (24 + 3 * lst + 24 + lst + 24 + 8 + 16), "flops": n * (pair + 40 * k)}
    if case["kind"] == "quench":
        step = n * (72.0 + 72.0 + 3 * lst + 24 + 8 + 16)
        return {"bytes": step * case["steps"] + n * (48 + 104),
                "flops": n * (pair + 40 * k) * case["steps"]}
    if case["kind"] == "fit":
        return {"bytes": n * (5 * lst + 5 * 24.0 + 24.0) + 2 * 24.0 * case["ntab"],
                "flops": n * k * 200.0}
    return {"bytes": n * (4 * lst + 4 * 24.0 + 72 + 24), "flops": n * k * 200.0}


# ------------------------------------------------------------------------------------------
# the same in plain numpy
# ------------------------------------------------------------------------------------------

def _tables(case):
    """Pair and embedding tables at knots 0..ntab+1 (zero at both ends), 64-bit."""
    n = case["ntab"]
    rc = CUNI_RC if case["alloy"] else W_RC
    csi = n / math.sqrt(rc)
    r = (np.arange(1, n + 1) * (1.0 / csi)) ** 2
    kinds = []
    if case["alloy"]:
        cu = (0.0855, 1.2240, 10.960, 2.2780, 3.615 * math.sqrt(0.5))
        ni = (0.0376, 1.0700, 16.999, 1.1890, 3.524 * math.sqrt(0.5))
        mix = tuple(math.sqrt(a * b) if k == 1 else 0.5 * (a + b)
                    for k, (a, b) in enumerate(zip(cu, ni)))
        # FPAIR order of PTYPE [[1, 3], [3, 2]]: Cu-Cu, Cu-Ni, Ni-Ni
        for a, xi, p, q, r0 in (cu, mix, ni):
            v = a * np.exp(-p * (r / r0 - 1.0))
            b = xi * xi * np.exp(-2.0 * q * (r / r0 - 1.0))
            kinds.append((v, 2.0 * v * (p / r0), b, b * (q / r0) * 2.0))
        kpair = np.array([[0, 1], [1, 2]])
    else:
        d = r - 3.25
        poly = 47.1346 - 33.7666 * r + 6.2542 * r * r
        v = np.where(r <= 3.25, 0.5 * d * d * poly, 0.0)
        dv = np.where(r <= 3.25, -(2.0 * d * poly + d * d * (-33.7666 + 2.0 * 6.2542 * r)), 0.0)
        d = r - 4.4002
        b = np.where(r <= 4.4002, 1.8964 ** 2 * d * d, 0.0)
        kinds.append((v, dv, b, np.where(r <= 4.4002, -1.8964 ** 2 * 2.0 * d, 0.0)))
        kpair = np.zeros((1, 1), int)
    z = np.zeros((len(kinds), n + 2))
    t = {"csi": csi, "rc": rc, "kpair": kpair, "potr": z.copy(), "fpotr": z.copy(),
         "potb": z.copy(), "fpotb": z.copy(), "eam": case["pot"] == "EAM_TYPE"}
    for k, (v, dv, b, db) in enumerate(kinds):
        t["potr"][k, 1:-1], t["fpotr"][k, 1:-1] = v * r, dv * r
        t["potb"][k, 1:-1], t["fpotb"][k, 1:-1] = b, db
    t["rhod"] = 20.0 * t["potb"].max() / n
    rho = np.arange(n) * t["rhod"]
    t["femb"], t["demb"] = np.zeros(n + 2), np.zeros(n + 2)
    with np.errstate(divide="ignore"):
        t["femb"][1:-1] = -np.sqrt(rho)
        t["demb"][1:-1] = np.where(rho > 0, -0.5 / np.sqrt(rho), 0.0)
    return t


def _half_pairs(b, rcut):
    """Pairs (i, j), each once, within rcut (minimum image)."""
    x, ln, per = b["x"], b["ln"], np.array(b["ifpd"], bool)
    n = len(x)

    def near(i, j):
        s = x[i] - x[j]
        s -= np.where(per & (np.abs(s) > 0.5 * ln), np.copysign(ln, s), 0.0)
        m = (s * s).sum(1) < rcut * rcut
        return i[m], j[m]

    nc = np.floor(ln / rcut).astype(int)
    if (nc < 3).any():
        got = [near(*(np.full(n - i - 1, i), np.arange(i + 1, n))) for i in range(n - 1)]
        return tuple(np.concatenate(p) for p in zip(*got))
    c3 = np.clip(((x - b["lo"]) / ln * nc).astype(int), 0, nc - 1)
    cell = (c3[:, 2] * nc[1] + c3[:, 1]) * nc[0] + c3[:, 0]
    order = np.argsort(cell, kind="stable")
    cnt = np.bincount(cell, minlength=nc.prod())
    start = np.concatenate([[0], np.cumsum(cnt)])
    got = []
    offs = [(a, c, d) for a in (-1, 0, 1) for c in (-1, 0, 1) for d in (-1, 0, 1)
            if (d, c, a) >= (0, 0, 0)]
    for a, c, d in offs:
        q = c3 + np.array([a, c, d])
        ok = (per | ((q >= 0) & (q < nc))).all(1)
        q = q % nc
        g = (q[:, 2] * nc[1] + q[:, 1]) * nc[0] + q[:, 0]
        m = np.where(ok, cnt[g], 0)
        i = np.repeat(np.arange(n), m)
        j = order[np.repeat(start[g], m) + np.arange(m.sum()) - np.repeat(np.cumsum(m) - m, m)]
        if (a, c, d) == (0, 0, 0):
            keep = i < j
            i, j = i[keep], j[keep]
        got.append(near(i, j))
    return tuple(np.concatenate(p) for p in zip(*got))


class _Exact:
    """Forces and energies of one box in numpy, over a pair list with room for the moves."""

    def __init__(self, b, t, room):
        self.b, self.t, self.n = b, t, len(b["x"])
        self.i, self.j = _half_pairs(b, t["rc"] + room)

    def pairs(self, x):
        b, t = self.b, self.t
        s = x[self.i] - x[self.j]
        per = np.array(b["ifpd"], bool)
        s -= np.where(per & (np.abs(s) > 0.5 * b["ln"]), np.copysign(b["ln"], s), 0.0)
        r2 = (s * s).sum(1)
        m = r2 <= t["rc"] ** 2
        i, j, s, r = self.i[m], self.j[m], s[m], np.sqrt(r2[m])
        sk = np.sqrt(r) * t["csi"]
        kk = np.minimum(sk.astype(int), t["potr"].shape[1] - 2)
        kind = t["kpair"][b["ityp"][i], b["ityp"][j]]
        return i, j, s, r, kind, kk, sk - kk

    @staticmethod
    def lerp(T, kind, kk, dk):
        a = T[kind, kk]
        return a + dk * (T[kind, kk + 1] - a)

    def both(self, i, j, a, c):
        return np.bincount(i, a, self.n) + np.bincount(j, c, self.n)

    def embed(self, rho):
        """F, F' and the derivatives of both with respect to rho, as the tables give them."""
        t = self.t
        some = rho > 0
        q = np.where(some, rho, 1.0)
        if not t["eam"]:
            f, d = -np.sqrt(q), -0.5 / np.sqrt(q)
            f1, d1 = d, 0.25 * q ** -1.5
        else:
            sk = q / t["rhod"] + 1.0
            kk = (sk + 1e-6).astype(int)
            df, dd = np.diff(t["femb"])[kk], np.diff(t["demb"])[kk]
            f, d = t["femb"][kk] + (sk - kk) * df, t["demb"][kk] + (sk - kk) * dd
            f1, d1 = df / t["rhod"], dd / t["rhod"]
        z = 0.0 * rho
        return (np.where(some, f, z), np.where(some, d, rho), np.where(some, f1, z),
                np.where(some, d1, z))

    def force(self, x):
        t = self.t
        p = i, j, s, r, kind, kk, dk = self.pairs(x)
        v = self.lerp(t["potb"], kind, kk, dk)
        rho = self.both(i, j, v, v)
        self.f_rho, d, _, _ = self.embed(rho)
        ft = (self.lerp(t["fpotr"], kind, kk, dk) / (r * r) +
              self.lerp(t["fpotb"], kind, kk, dk) * (d[i] + d[j]) / r)
        self.last, self.ft, self.rho, self.d = p, ft, rho, d
        w = ft[:, None] * s
        return np.stack([self.both(i, j, w[:, k], -w[:, k]) for k in range(3)], 1)

    def epot(self):
        i, j, s, r, kind, kk, dk = self.last
        v = self.lerp(self.t["potr"], kind, kk, dk) / r
        return self.both(i, j, v, v) + self.f_rho


def _exact_md(case, b, t):
    h = 2.0 if case["alloy"] else 1.0
    e = _Exact(b, t, 1.0)
    im = 1.0 / b["mass"][b["ityp"]][:, None]
    x, v, dis = b["x"].copy(), b["v"].copy(), np.zeros_like(b["x"])
    per, lo, hi, ln = np.array(b["ifpd"], bool), b["lo"], b["lo"] + b["ln"], b["ln"]
    f = e.force(x)
    for k in range(case["steps"]):
        d = h * v + 0.5 * h * h * f * im
        x, dis = x + d, dis + d
        x = np.where(per & (x > hi), x - ln, np.where(per & (x < lo), x + ln, x))
        v = v + 0.5 * h * f * im
        f = e.force(x)
        v = v + 0.5 * h * f * im
    return x, v, f, dis


def _exact_fit(case, seed, raw):
    """Loss and gradient: tables linear in the coefficients, every pair a lerp of them."""
    t0 = _tables(case)
    n, eam, csi, rhod = case["ntab"], t0["eam"], t0["csi"], t0["rhod"]
    c, target = _coefficients(case, seed)
    k = np.arange(1, n + 1)
    r = (k / csi) ** 2

    def val(y):
        p = np.pad(y, 1)
        return (p[:-2] + 4.0 * p[1:-1] + p[2:]) / 6.0

    def slope(y):
        p = np.pad(y, 1)
        return 0.5 * (p[2:] - p[:-2])

    def slope_t(y):
        return -slope(y)

    def tables(c):
        t = dict(t0)
        t["potr"], t["fpotr"] = np.pad(val(c[0]) * r, 1)[None], np.pad(-k * slope(c[0]), 1)[None]
        t["potb"] = np.pad(val(c[1]), 1)[None]
        t["fpotb"] = np.pad(-slope(c[1]) * csi * csi / (2.0 * k), 1)[None]
        if eam:
            t["femb"], t["demb"] = np.pad(val(c[2]), 1), np.pad(slope(c[2]) / rhod, 1)
        return t

    tc, tt = tables(c), tables(target)
    atoms, nb = sum(len(b["x"]) for b in raw), len(raw)
    loss, g = 0.0, {q: np.zeros(n + 2) for q in ("potr", "fpotr", "potb", "fpotb", "femb", "demb")}

    def into(q, kk, dk, w):
        g[q] += np.bincount(kk, w * (1.0 - dk), n + 2) + np.bincount(kk + 1, w * dk, n + 2)

    for b in raw:
        e, w = _Exact(b, tc, 0.0), _Exact(b, tt, 0.0)
        df = e.force(b["x"]) - w.force(b["x"])
        nat = len(b["x"])
        de = (e.epot().sum() - w.epot().sum()) / nat
        loss += (df * df).sum() / atoms + 0.1 * de * de / nb
        G, gb = 2.0 * df / atoms, 0.2 * de / (nat * nb)
        i, j, s, rr, kind, kk, dk = e.last
        gs = ((G[i] - G[j]) * s).sum(1)              # both directions of the pair
        into("fpotr", kk, dk, gs / (rr * rr))
        into("potr", kk, dk, 2.0 * gb / rr)
        into("fpotb", kk, dk, gs * (e.d[i] + e.d[j]) / rr)
        lam = e.both(i, j, *(2 * [gs * e.lerp(tc["fpotb"], kind, kk, dk) / rr]))
        _, _, f1, d1 = e.embed(e.rho)
        mu = lam * d1 + gb * f1
        into("potb", kk, dk, mu[i] + mu[j])
        if eam:
            some = e.rho > 0
            sk = e.rho[some] / rhod + 1.0
            ke = (sk + 1e-6).astype(int)
            into("demb", ke, sk - ke, lam[some])
            into("femb", ke, sk - ke, np.full(some.sum(), gb))
    g = {q: v[1:-1] for q, v in g.items()}
    grad = np.zeros((3, n))
    grad[0] = val(g["potr"] * r) + slope_t(-k * g["fpotr"])
    grad[1] = val(g["potb"]) + slope_t(-g["fpotb"] * csi * csi / (2.0 * k))
    if eam:
        grad[2] = val(g["femb"]) + slope_t(g["demb"] / rhod)
    return {"loss": float(loss), "grad": grad}


def exact(case, seed):
    n = _atoms(case)
    if n * (3.0 if case["alloy"] else 1.0) * case["steps"] > 2.5e6:
        return None
    raw, t = _inputs(case, seed), _tables(case)
    if case["kind"] == "fit":
        return _exact_fit(case, seed, raw)
    if case["kind"] == "md":
        x, v, f, dis = (np.concatenate(q) for q in zip(*(_exact_md(case, b, t) for b in raw)))
        return {"x": x, "v": v, "f": f, "statu": None, "dis": dis}
    if case["kind"] == "stress":
        b = raw[0]
        e = _Exact(b, t, 0.0)
        f = e.force(b["x"])
        i, j, s = e.last[:3]
        w = [e.ft * s[:, a] * s[:, c] for a in range(3) for c in range(3)]
        avp = np.stack([e.both(i, j, q, q) for q in w], 1)
        return {"avp": avp, "vir": 0.5 * avp.sum(0).reshape(3, 3), "f": f}
    if case["kind"] == "quench":
        return None   # which component stops when depends on the sign of a product
    rng = np.random.default_rng([seed, 22])
    b = raw[0]
    x = b["x"] + rng.normal(0.0, 0.03, b["x"].shape)
    per, lo, ln = np.array(b["ifpd"], bool), b["lo"], b["ln"]
    b["x"] = np.where(per & (x < lo), x + ln, np.where(per & (x >= lo + ln), x - ln, x))
    e = _Exact(b, t, 0.0)
    f = e.force(b["x"])
    ep = e.epot()
    return {"f": f, "epot": ep, "e": np.array([ep.sum()])}
