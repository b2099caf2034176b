"""Performance cases: the calls that a user of libmdx makes, from the smallest to the largest.

Five ways into the library, each over its range of sizes:

  step     one Pair::compute of a host program that integrates by itself (pair_style lj/cut/mdx, eam/mdx):
           positions in from host memory, forces out to it; `reneigh` steps also hand the atoms over and build the
           neighbour list, as a host program does whenever it reneighbours; `peratom` steps also return the
           per-atom energies and virials that dumps and computes read
  device   the same on positions that already lie in device memory (Context.compute_noalloc), list included
  run      a stretch of molecular dynamics that stays on the device (Context.run), then the state read back
  batch    forces and energies of many small configurations whose positions have just changed
  fit      loss and parameter gradient of force matching over many configurations (PyTorch autograd)

Systems are those of the benchmark and the tests: the lj/cut melt (fcc at reduced density 0.8442, T = 1.44, cutoff 2.5),
the Kob-Andersen 80:20 mixture (density 1.2), fcc copper (Cu_u3.eam, 1600 K) and free copper-like clusters with a
64-knot eam.  Inputs come from the seed alone; `exact` restates each pass in FP64 with plain torch.
"""
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CU = os.path.join(ROOT, "tests", "golden", "Cu_u3.eam")

BOLTZ, MVV2E = 8.617343e-5, 1.0364269e-4  # metal units
LJ_PAIRS = {(1, 1): (1.0, 1.0, 2.5)}
KA_PAIRS = {(1, 1): (1.0, 1.0, 2.5), (1, 2): (1.5, 0.8, 2.0), (2, 2): (0.5, 0.88, 2.2)}
FCC = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
SC = np.zeros((1, 3))
# lattice constant, basis, masses, temperature in velocity^2 * mass, skin, neigh_modify (every, delay), time step
STYLES = {
    "lj": dict(a=(4.0 / 0.8442) ** (1.0 / 3.0), basis=FCC, mass=[0.0, 1.0], mv2=1.44, skin=0.3, every=20, delay=0,
               dt=0.005, ftm2v=1.0, cut=2.5, noise=0.02),
    "ka": dict(a=(1.0 / 1.2) ** (1.0 / 3.0), basis=SC, mass=[0.0, 1.0, 1.0], mv2=0.8, skin=0.3, every=1, delay=0,
               dt=0.002, ftm2v=1.0, cut=2.5, noise=0.02),
    "eam": dict(a=3.615, basis=FCC, mass=[0.0, 63.55], mv2=BOLTZ * 1600.0 / MVV2E, skin=1.0, every=1, delay=5,
                dt=0.005, ftm2v=1.0 / MVV2E, cut=4.95, noise=0.05),
}
CLUSTER_CUT, CLUSTER_KNOTS = 4.95, 64


def listed():
    return [
        # a host program's time step on a system of a few hundred atoms: latency only
        dict(name="step_lj_500", kind="step", style="lj", precision="fp64", cx=5, cy=5, cz=5, reneigh=False,
             peratom=False),
        # a host program's reneighbouring step that also writes a dump, bench-sized copper with uneven sides
        dict(name="reneigh_eam_108k", kind="step", style="eam", precision="fp64", cx=29, cy=31, cz=30, reneigh=True,
             peratom=True),
        # a program that keeps its atoms in device memory, near the largest size that entry point takes
        dict(name="device_lj_32k", kind="device", style="lj", precision="mixed", cx=20, cy=20, cz=20),
        # equilibration of a glass former, the preparation of the force-matching data: small, two types
        dict(name="run_ka_8k", kind="run", style="ka", precision="fp64", cx=20, cy=20, cz=20, steps=100),
        # the lj/cut and eam benchmark inputs at their own size (32,000 atoms, 100 steps)
        dict(name="run_lj_32k", kind="run", style="lj", precision="mixed", cx=20, cy=20, cz=20, steps=100),
        dict(name="run_eam_32k", kind="run", style="eam", precision="fp64", cx=20, cy=20, cz=20, steps=100),
        # the benchmark's scaled sizes, and a ragged one between them in full precision
        dict(name="run_eam_256k", kind="run", style="eam", precision="mixed", cx=40, cy=40, cz=40, steps=100),
        dict(name="run_lj_508k", kind="run", style="lj", precision="fp64", cx=47, cy=53, cz=51, steps=100),
        dict(name="run_lj_2048k", kind="run", style="lj", precision="mixed", cx=80, cy=80, cz=80, steps=100),
        # forces of an ensemble of small periodic boxes after a move of all of them
        dict(name="batch_ka_96x1331", kind="batch", style="ka", precision="fp64", replicas=96, cells=11),
        # force matching at the benchmark's sizes: snapshots of one system, and clusters of uneven size
        dict(name="fit_ka_64x8000", kind="fit", style="ka", precision="mixed", replicas=64, cells=20),
        dict(name="fit_eam_512", kind="fit", style="eam", precision="mixed", replicas=512, atoms=5000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cells(rng, style, lo, hi):
    """Uneven cell counts of a box with about lo..hi atoms (spread over the logarithm)."""
    per = len(STYLES[style]["basis"])
    least = math.ceil(2.02 * (STYLES[style]["cut"] + STYLES[style]["skin"]) / STYLES[style]["a"])
    side = (math.exp(rng.uniform(math.log(lo), math.log(hi))) / per) ** (1.0 / 3.0)
    return {k: max(least, int(round(side * rng.uniform(0.85, 1.15)))) for k in ("cx", "cy", "cz")}


def draw(rng):
    kind = rng.choice(["step", "step", "device", "run", "run", "run", "batch", "fit"])
    style = rng.choice(["lj", "ka", "eam"])
    case = dict(kind=kind, style=style, precision=rng.choice(["fp64", "mixed"]))
    if kind == "step":
        case.update(_cells(rng, style, 300, 700000), reneigh=rng.random() < 0.4, peratom=rng.random() < 0.3)
    elif kind == "device":
        case.update(_cells(rng, style, 300, 20000))
    elif kind == "run":
        case.update(_cells(rng, style, 500, 300000 if style == "eam" else 800000), steps=rng.choice([50, 100, 150]))
    elif style == "eam":
        case.update(replicas=_log_int(rng, 2, 400), atoms=_log_int(rng, 300, 5000))
    else:
        case["style"] = "ka"
        case.update(replicas=_log_int(rng, 2, 64), cells=rng.randint(8, 20))
    return case


# ------------------------------------------------------------------ inputs

def _rng(case, seed):
    return np.random.default_rng([int(seed), 77])


def _types(rng, style, n):
    t = np.ones(n, dtype=np.int32)
    if style == "ka":
        t[rng.permutation(n)[:n // 5]] = 2
    return t


def _system(case, seed):
    """Box, positions, velocities and types of one periodic system."""
    s, rng = STYLES[case["style"]], _rng(case, seed)
    n3 = [case["cx"], case["cy"], case["cz"]]
    k, j, i, b = np.meshgrid(*[np.arange(q) for q in n3[::-1]], np.arange(len(s["basis"])), indexing="ij")
    cells = np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1).astype(np.float64)
    hi = np.array(n3, dtype=np.float64) * s["a"]
    x = (cells + s["basis"][b.ravel()]) * s["a"] + rng.normal(0.0, s["noise"], cells.shape)
    x -= hi * np.floor(x / hi)
    n = len(x)
    t = _types(rng, case["style"], n)
    v = rng.normal(0.0, 1.0, x.shape) * np.sqrt(s["mv2"] / np.array([1.0] + s["mass"][1:])[t])[:, None]
    v -= v.mean(axis=0)
    return dict(n=n, lo=np.zeros(3), hi=hi, x=np.minimum(x, np.nextafter(hi, 0.0)), v=v, types=t, rng=rng)


def _moved(case, sysm):
    """The positions a few steps after the list was built: every atom well within half the skin."""
    lim = 0.2 * STYLES[case["style"]]["skin"]
    return sysm["x"] + sysm["rng"].uniform(-lim, lim, sysm["x"].shape)


def _fcc_sites(n):
    """The n fcc sites nearest the origin."""
    m = int(math.ceil((n / 4.0) ** (1.0 / 3.0))) + 2
    r = np.arange(-m, m + 1)
    k, j, i = np.meshgrid(r, r, r, indexing="ij")
    sites = ((np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1)[:, None, :] + FCC[None]) * 3.615).reshape(-1, 3)
    return sites[np.argsort(np.sum(sites ** 2, axis=1), kind="stable")[:n]]


def _replicas(case, seed):
    """Boxes, positions and types of many configurations, in one array."""
    rng, nrep = _rng(case, seed), case["replicas"]
    if case["style"] == "ka":
        s, c = STYLES["ka"], case["cells"]
        k, j, i = np.meshgrid(*[np.arange(c)] * 3, indexing="ij")
        sites = np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1) * s["a"]
        n = len(sites)
        x = np.tile(sites, (nrep, 1)) + rng.normal(0.0, 0.04, (nrep * n, 3))
        t = np.concatenate([_types(rng, "ka", n) for _ in range(nrep)])
        lo, hi = np.zeros((nrep, 3)), np.full((nrep, 3), c * s["a"])
        x -= hi[0] * np.floor(x / hi[0])
        return dict(natoms=np.full(nrep, n), lo=lo, hi=hi, periodic=np.ones((nrep, 3), np.int32),
                    x=np.minimum(x, np.nextafter(hi[0], 0.0)), types=t, ntypes=2, rng=rng)
    sites = _fcc_sites(case["atoms"])
    # the sizes belong to the case, the positions to the seed
    natoms = np.random.default_rng(7).integers(max(50, case["atoms"] // 25), case["atoms"] + 1, nrep)
    x = np.concatenate([sites[:q] for q in natoms])
    x = x + rng.normal(0.0, 0.08, x.shape)
    starts = np.concatenate([[0], np.cumsum(natoms)[:-1]])
    lo = np.minimum.reduceat(x, starts) - 8.0
    hi = np.maximum.reduceat(x, starts) + 8.0
    return dict(natoms=natoms, lo=lo, hi=hi, periodic=np.zeros((nrep, 3), np.int32), x=x,
                types=np.ones(len(x), np.int32), ntypes=1, rng=rng)


def _cluster_knots(rng):
    """Knot values of the clusters' eam (embedding, density, r * pair term), each within a percent of the analytic
    form, as a fit in progress holds them."""
    re, n = 3.615 / math.sqrt(2.0), CLUSTER_KNOTS
    dr = CLUSTER_CUT / (n - 1)
    r = np.arange(n) * dr
    dens = np.exp(-6.0 * (r / re - 1.0))
    shells = zip((12, 6, 24, 12), (0.5, 1.0, 1.5, 2.0))
    rho_e = sum(q * math.exp(-6.0 * (3.615 * math.sqrt(d) / re - 1.0)) for q, d in shells if 3.615 * math.sqrt(d) < CLUSTER_CUT)
    drho = 2.0 * rho_e / (n - 1)
    frho = -3.0 * np.sqrt(np.arange(n) * drho / rho_e)
    z2r = 27.2 * 0.529 * (11.0 * np.exp(-1.5 * r)) ** 2
    return drho, dr, [k * (1.0 + rng.uniform(-0.01, 0.01, n)) for k in (frho, dens, z2r)]


def _fit_inputs(case, seed):
    """Configurations, starting parameters and target forces of one fit."""
    g = _replicas(case, seed)
    rng = g["rng"]
    if case["style"] == "ka":
        keys = [(1, 1), (1, 2), (2, 2)]
        par = [np.array([KA_PAIRS[k][q] for k in keys]) * (1.0 + rng.uniform(-0.02, 0.02, 3)) for q in (0, 1)]
        g.update(par=par, cut=np.array([KA_PAIRS[k][2] for k in keys]), target=rng.normal(0.0, 20.0, g["x"].shape))
    else:
        drho, dr, par = _cluster_knots(rng)
        g.update(par=par, drho=drho, dr=dr, cut=CLUSTER_CUT, target=rng.normal(0.0, 1.0, g["x"].shape))
    return g


# ------------------------------------------------------------------ prepare, run

def _pair_style(ctx, mdx, style):
    if style == "eam":
        mdx.eam_context_tables(ctx, CU)
    else:
        pairs = KA_PAIRS if style == "ka" else LJ_PAIRS
        ctx.pair_lj_from_coeffs(len(STYLES[style]["mass"]) - 1, pairs)


def _context(case, sysm, mdx):
    s = STYLES[case["style"]]
    ctx = mdx.Context(0)
    ctx.set_box(sysm["lo"], sysm["hi"], (1, 1, 1))
    if case["kind"] != "device":
        ctx.set_atoms(sysm["x"], sysm["types"], np.array(s["mass"]), v=sysm["v"])
    _pair_style(ctx, mdx, case["style"])
    ctx.neigh_modify(s["skin"], every=s["every"], delay=s["delay"], check=True)
    ctx.precision(mdx.MIXED if case["precision"] == "mixed" else mdx.FP64)
    return ctx


def prepare(case, seed):
    from lammps_amd import mdx
    kind = case["kind"]
    st = dict(case=case, kind=kind)
    if kind in ("step", "device", "run"):
        sysm = _system(case, seed)
        st.update(n=sysm["n"], ctx=_context(case, sysm, mdx))
    if kind == "step":
        st.update(x=_moved(case, sysm), types=sysm["types"], mass=np.array(STYLES[case["style"]]["mass"]))
        if not case["reneigh"]:
            st["ctx"].neigh_build()
    elif kind == "device":
        st.update(x=torch.tensor(sysm["x"], device="cuda"), types=torch.tensor(sysm["types"], device="cuda"),
                  f=torch.zeros((sysm["n"], 3), dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
    elif kind == "run":
        st["ctx"].setup()
        n = sysm["n"]
        st["host"] = [np.zeros((n, 3)), np.zeros((n, 3)), np.zeros((n, 3)), np.zeros((n, 3), dtype=np.int32)]
    elif kind == "batch":
        from lammps_amd import batch as B
        if case["style"] == "ka":
            g = _replicas(case, seed)
        else:
            g = _fit_inputs(case, seed)
        b = B.Batch(g["natoms"], g["lo"], g["hi"], g["periodic"], g["ntypes"], g["types"])
        b.precision(B.MIXED if case["precision"] == "mixed" else B.FP64)
        if case["style"] == "ka":
            eps, sig, cut = (_table([KA_PAIRS[k][q] for k in ((1, 1), (1, 2), (2, 2))]) for q in range(3))
            b.lj_init(eps, sig, cut)
        else:
            b.eam_init(g["drho"], g["dr"], g["cut"], *g["par"])
        st.update(batch=b, x=torch.tensor(g["x"], device="cuda"),
                  f=torch.zeros((len(g["x"]), 3), dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
    elif kind == "fit":
        from lammps_amd import batch as B
        from lammps_amd import fit
        g = _fit_inputs(case, seed)
        prec = B.MIXED if case["precision"] == "mixed" else B.FP64
        if case["style"] == "ka":
            fm = fit.LJForceMatch(g["natoms"], g["lo"], g["hi"], g["periodic"], 2, g["types"], g["x"], g["cut"],
                                  precision=prec)
        else:
            fm = fit.EAMForceMatch(g["natoms"], g["lo"], g["hi"], g["periodic"], g["x"], g["drho"], g["dr"], g["cut"],
                                   precision=prec)
        st.update(fm=fm, par=[torch.tensor(p, requires_grad=True) for p in g["par"]],
                  target=torch.tensor(g["target"], device="cuda"))
        torch.cuda.synchronize()
    return st


def _table(v):
    return np.array([[0.0, 0.0, 0.0], [0.0, v[0], v[1]], [0.0, v[1], v[2]]])


def run(st):
    case, kind = st["case"], st["kind"]
    if kind == "step":
        ctx = st["ctx"]
        if case["reneigh"]:
            ctx.set_atoms(st["x"], st["types"], st["mass"])
            ctx.neigh_build()
            return ctx.compute(3, 5, peratom=True) if case["peratom"] else ctx.compute(1, 1)
        ctx.set_positions(st["x"])
        return ctx.compute(3, 5, peratom=True) if case["peratom"] else ctx.compute(0, 0)["f"]
    if kind == "device":
        st["f"].zero_()
        torch.cuda.current_stream().synchronize()
        e, w = st["ctx"].compute_noalloc(st["n"], st["x"].data_ptr(), st["types"].data_ptr(), st["f"].data_ptr(), 1, 1)
        return dict(f=st["f"], eng=e, virial=w)
    if kind == "run":
        from lammps_amd import mdx
        s, ctx = STYLES[case["style"]], st["ctx"]
        rows = ctx.run(case["steps"], s["dt"], s["ftm2v"])
        x, v, f, image = st["host"]
        # the state into the program's own arrays, as a host program keeps them (mdx_get_atoms)
        rc = mdx.lib().mdx_get_atoms(ctx.h, *[mdx._ptr(a) for a in (x, v, f)], mdx._ptr(image, mdx._ip))
        if rc != mdx.OK:
            raise mdx.MdxError(rc, mdx.lib().mdx_last_error().decode())
        return dict(x=x, v=v, f=f, image=image, thermo=np.array(rows[-1][1]))
    if kind == "batch":
        b = st["batch"]
        b.set_positions(st["x"])
        _, e = b.lj_forces(out=st["f"]) if case["style"] == "ka" else b.eam_forces(out=st["f"])
        return dict(f=st["f"], energy=e)
    for p in st["par"]:
        p.grad = None
    force = st["fm"](*st["par"])
    loss = ((force - st["target"]) ** 2).sum() / (3.0 * force.shape[0])
    loss.backward()
    return dict(f=force.detach(), loss=loss.detach(), grad=[p.grad for p in st["par"]])


# ------------------------------------------------------------------ work

def _atoms(case):
    if "cx" in case:
        return case["cx"] * case["cy"] * case["cz"] * len(STYLES[case["style"]]["basis"])
    return case["replicas"] * (case["cells"] ** 3 if case["style"] == "ka" else int(0.52 * case["atoms"]))


def work(case):
    """Bytes and operations of one pass that no implementation avoids: inputs read once, outputs written once (a run
    reads and writes positions and velocities at every step), each pair within the cutoff evaluated once."""
    n, kind, eam = _atoms(case), case["kind"], case["style"] == "eam"
    density = 4.0 / 3.615 ** 3 if eam else 1.2 if case["style"] == "ka" else 0.8442
    pairs = 0.5 * n * density * 4.18879 * STYLES[case["style"]]["cut"] ** 3
    flops = pairs * (90.0 if eam else 33.0)
    if kind == "run":
        return dict(bytes=case["steps"] * n * 96.0 + n * 84.0, flops=case["steps"] * (flops + 18.0 * n))
    if kind == "fit":
        return dict(bytes=n * (24.0 + 24.0 + 24.0 + 24.0), flops=flops * 2.5)
    return dict(bytes=n * (52.0 + (56.0 if case.get("peratom") else 0.0)), flops=flops)


# ------------------------------------------------------------------ the same in 64 bits, in plain torch

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _brute(x, prd, periodic, cut):
    """Pairs i < j within cut of one small configuration."""
    n = len(x)
    d2 = torch.zeros((n, n), dtype=torch.float64, device=x.device)
    for k in range(3):
        d = x[:, None, k] - x[None, :, k]
        if periodic[k]:
            d -= prd[k] * torch.round(d / prd[k])
        d2 += d * d
    return torch.nonzero(torch.triu(d2 <= cut * cut, diagonal=1), as_tuple=True)


def _pairs(x, prd, cut):
    """Pairs i < j (each once) within cut of a periodic system, x in [0, prd): a cell list over 14 half offsets."""
    nb = [int(p / cut) for p in prd]
    if min(nb) < 3:
        return _brute(x, prd, (1, 1, 1), cut)
    dev = x.device
    size = torch.tensor([p / q for p, q in zip(prd, nb)], dtype=torch.float64, device=dev)
    top = torch.tensor(nb, device=dev) - 1
    c = torch.minimum((x / size).long(), top)
    key = (c[:, 2] * nb[1] + c[:, 1]) * nb[0] + c[:, 0]
    order = torch.argsort(key)
    xs, cs = x[order], c[order]
    count = torch.bincount(key, minlength=nb[0] * nb[1] * nb[2])
    start = torch.cumsum(count, 0) - count
    left, right = [], []
    offsets = [(a, b, d) for d in (-1, 0, 1) for b in (-1, 0, 1) for a in (-1, 0, 1) if (d, b, a) >= (0, 0, 0)]
    step = 400000
    for a, b, d in offsets:
        for i0 in range(0, len(x), step):
            q = cs[i0:i0 + step]
            other = ((((q[:, 2] + d) % nb[2]) * nb[1] + (q[:, 1] + b) % nb[1]) * nb[0] + (q[:, 0] + a) % nb[0])
            m = count[other]
            i = torch.repeat_interleave(torch.arange(i0, i0 + len(q), device=dev), m)
            j = torch.arange(len(i), device=dev) - torch.repeat_interleave(torch.cumsum(m, 0) - m, m)
            j += torch.repeat_interleave(start[other], m)
            r2 = torch.zeros(len(i), dtype=torch.float64, device=dev)
            for k in range(3):
                e = xs[i, k] - xs[j, k]
                r2 += (e - prd[k] * torch.round(e / prd[k])) ** 2
            keep = r2 <= cut * cut
            if (a, b, d) == (0, 0, 0):
                keep &= j > i
            left.append(order[i[keep]])
            right.append(order[j[keep]])
    return torch.cat(left), torch.cat(right)


def _spline(knots, delta):
    """PairEAM's interpolation: value and derivative as functions of the position (knot 1 at 0)."""
    f, n = knots, len(knots)
    s = [f[1] - f[0], 0.5 * (f[2] - f[0])]
    s += [((f[m - 2] - f[m + 2]) + 8.0 * (f[m + 1] - f[m - 1])) / 12.0 for m in range(2, n - 2)]
    s = torch.stack(s + [0.5 * (f[n - 1] - f[n - 3]), f[n - 1] - f[n - 2]])
    up, df = s[1:], f[1:] - f[:-1]
    c4 = 3.0 * df - 2.0 * s[:-1] - up
    c3 = s[:-1] + up - 2.0 * df

    def at(u, low):
        p = u / delta + 1.0
        m = torch.clamp(p.long(), 1 if low else 0, n - 1)
        p = torch.clamp(p - m, max=1.0)
        m = m - 1
        a, b, c, d = c3[m], c4[m], s[m], f[m]
        return ((a * p + b) * p + c) * p + d, ((3.0 * a * p + 2.0 * b) * p + c) / delta
    return at


def _funcfl(path):
    """Knots of a funcfl file (PairEAM drops the last point): embedding, density, r * pair term."""
    with open(path) as fh:
        lines = fh.read().split("\n")
    nrho, drho, nr, dr = (float(q) for q in lines[2].split()[:4])
    nrho, nr = int(nrho), int(nr)
    v = np.array(" ".join(lines[3:]).split(), dtype=np.float64)
    z, rho = v[nrho:nrho + nr - 1], v[nrho + nr:nrho + 2 * nr - 1]
    return drho, dr, [v[:nrho - 1], rho, 27.2 * 0.529 * z * z], (nrho - 1) * drho


def _lj_terms(style, par, dev):
    keys = [(1, 1), (1, 2), (2, 2)]
    pairs = KA_PAIRS if style == "ka" else {k: LJ_PAIRS[(1, 1)] for k in keys}
    eps, sig = par if par is not None else (torch.tensor([pairs[k][q] for k in keys], dtype=torch.float64, device=dev)
                                            for q in (0, 1))
    return eps, sig, torch.tensor([pairs[k][2] for k in keys], dtype=torch.float64, device=dev)


class _Potential:
    """Forces (and energies, virials) of pairs (i, j) with separations del = x_i - x_j, in FP64."""

    def __init__(self, style, par=None, drho=None, dr=None):
        self.eam, dev = style == "eam", _device()
        if not self.eam:
            self.eps, self.sig, self.cut = _lj_terms(style, par, dev)
            self.cutmax = float(self.cut.max())
            return
        if par is None:
            drho, dr, knots, self.rhomax = _funcfl(CU)
            par = [torch.tensor(k, device=dev) for k in knots]
        else:
            self.rhomax = (len(par[0]) - 1) * drho
        self.frho, self.rhor, self.z2r = _spline(par[0], drho), _spline(par[1], dr), _spline(par[2], dr)
        self.cutmax = CLUSTER_CUT

    def __call__(self, n, i, j, d, types, tally=True):
        """(f, eatom, vatom) of n atoms; vatom rows xx yy zz xy xz yz."""
        r2 = (d * d).sum(1)
        if self.eam:
            keep = r2 < self.cutmax ** 2
        else:
            t = types[i] + types[j] - 2
            keep = r2 < self.cut[t] ** 2
            t = t[keep]
        i, j, d, r2 = i[keep], j[keep], d[keep], r2[keep]
        zero = torch.zeros(n, dtype=torch.float64, device=d.device)
        if self.eam:
            r = torch.sqrt(r2)
            dens, ddens = self.rhor(r, False)
            rho = zero.index_add(0, i, dens).index_add(0, j, dens)
            emb, fp = self.frho(rho, True)
            z2, dz2 = self.z2r(r, False)
            phi = z2 / r
            fpair = -((fp[i] + fp[j]) * ddens + dz2 / r - phi / r) / r
            emb = emb + torch.where(rho > self.rhomax, fp * (rho - self.rhomax), zero)
        else:
            s6 = self.sig[t] ** 6 / r2 ** 3
            fpair = 24.0 * self.eps[t] * s6 * (2.0 * s6 - 1.0) / r2
            phi, emb = 4.0 * self.eps[t] * s6 * (s6 - 1.0), zero
        fd = fpair[:, None] * d
        f = torch.zeros((n, 3), dtype=torch.float64, device=d.device).index_add(0, i, fd).index_add(0, j, -fd)
        if not tally:
            return f, None, None
        e = emb + 0.5 * zero.index_add(0, i, phi).index_add(0, j, phi)
        w = 0.5 * torch.stack([d[:, a] * fd[:, b] for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))], 1)
        v = torch.zeros((n, 6), dtype=torch.float64, device=d.device).index_add(0, i, w).index_add(0, j, w)
        return f, e, v


def _sep(x, i, j, prd):
    d = x[i] - x[j]
    return d - prd * torch.round(d / prd)


def _exact_run(case, seed):
    """Velocity Verlet with the list rebuilt when LAMMPS rebuilds it (every, delay, check yes)."""
    s, q, dev = STYLES[case["style"]], _system(case, seed), _device()
    x, v = torch.tensor(q["x"], device=dev), torch.tensor(q["v"], device=dev)
    types, prd = torch.tensor(q["types"], device=dev).long(), torch.tensor(q["hi"], device=dev)
    pot, n = _Potential(case["style"]), q["n"]
    mass = torch.tensor(s["mass"], dtype=torch.float64, device=dev)[types][:, None]
    # the list holds a pair up to its own type pair's cutoff plus the skin
    def build(x):
        i, j = _pairs(x, q["hi"].tolist(), s["cut"] + s["skin"])
        if not pot.eam:
            d = _sep(x, i, j, prd)
            keep = (d * d).sum(1) <= (pot.cut[types[i] + types[j] - 2] + s["skin"]) ** 2
            i, j = i[keep], j[keep]
        return i, j
    i, j = build(x)
    hold, ago = x.clone(), 0
    f, _, _ = pot(n, i, j, _sep(x, i, j, prd), types, False)
    half = 0.5 * s["dt"] * s["ftm2v"] / mass
    for k in range(case["steps"]):
        v = v + half * f
        x = x + s["dt"] * v
        ago += 1
        if ago >= s["delay"] and ago % s["every"] == 0 and float(((x - hold) ** 2).sum(1).max()) > (0.5 * s["skin"]) ** 2:
            x = torch.where(x < 0, x + prd, x)
            x = torch.where(x >= prd, x - prd, x)
            i, j = build(x)
            hold, ago = x.clone(), 0
        f, e, w = pot(n, i, j, _sep(x, i, j, prd), types, k == case["steps"] - 1)
        v = v + half * f
    mv2 = (mass * v * v).sum()
    return dict(x=x, v=v, f=f, image=None, thermo=torch.cat([mv2[None], e.sum()[None], w.sum(0)]))


def _exact_replicas(g, pot):
    """Forces and energies of every replica, pairs by brute force."""
    dev, at, fs, es = _device(), 0, [], []
    for r, n in enumerate(g["natoms"]):
        n = int(n)
        x, types = torch.tensor(g["x"][at:at + n], device=dev), torch.tensor(g["types"][at:at + n], device=dev).long()
        prd, per = torch.tensor(g["hi"][r] - g["lo"][r], device=dev), g["periodic"][r]
        i, j = _brute(x, prd, per, pot.cutmax)
        d = _sep(x, i, j, prd) if per[0] else x[i] - x[j]
        f, e, _ = pot(n, i, j, d, types)
        fs.append(f)
        es.append(e.sum())
        at += n
    return torch.cat(fs), torch.stack(es)


def _exact_fit(case, seed):
    g, dev = _fit_inputs(case, seed), _device()
    par = [torch.tensor(p, device=dev, requires_grad=True) for p in g["par"]]
    # one replica's graph at a time: loss and gradient are sums over the replicas
    n, at, fs, loss = len(g["x"]), 0, [], 0.0
    for r, m in enumerate(g["natoms"]):
        one = {k: g[k][r:r + 1] for k in ("natoms", "lo", "hi", "periodic")}
        one.update(x=g["x"][at:at + m], types=g["types"][at:at + m])
        pot = _Potential(case["style"], par, g.get("drho"), g.get("dr"))
        f, _ = _exact_replicas(one, pot)
        part = ((f - torch.tensor(g["target"][at:at + m], device=dev)) ** 2).sum() / (3.0 * n)
        part.backward()
        fs.append(f.detach())
        loss = loss + part.detach()
        at += m
    return dict(f=torch.cat(fs), loss=loss, grad=[p.grad for p in par])


def exact(case, seed):
    kind = case["kind"]
    if kind == "run":
        return _exact_run(case, seed) if _atoms(case) * case["steps"] <= 60_000_000 else None
    if kind == "fit":
        return _exact_fit(case, seed)
    if kind == "batch":
        if case["style"] == "ka":
            f, e = _exact_replicas(_replicas(case, seed), _Potential("ka"))
        else:
            g, dev = _fit_inputs(case, seed), _device()
            par = [torch.tensor(p, device=dev) for p in g["par"]]
            f, e = _exact_replicas(g, _Potential("eam", par, g["drho"], g["dr"]))
        return dict(f=f, energy=e)
    q, dev = _system(case, seed), _device()
    x = torch.tensor(_moved(case, q) if kind == "step" else q["x"], device=dev)
    prd, types, pot = torch.tensor(q["hi"], device=dev), torch.tensor(q["types"], device=dev).long(), _Potential(case["style"])
    xw = x - prd * torch.floor(x / prd)
    i, j = _pairs(xw, q["hi"].tolist(), pot.cutmax)
    f, e, w = pot(q["n"], i, j, _sep(x, i, j, prd), types)
    if kind == "device":
        return dict(f=f, eng=float(e.sum()), virial=w.sum(0))
    if not (case["reneigh"] or case["peratom"]):
        return f
    return dict(f=f, eng=float(e.sum()), virial=w.sum(0), eatom=e if case["peratom"] else None,
                vatom=w if case["peratom"] else None)
