"""Batched forces and force-matching adjoints on the device (mdx_batch.h)
against the FP64 oracle (oracle/fitref.c, pinned by finite differences in
tests/test_fit_oracle.py).

Tolerances: FP64 forces max_rel <= 1e-11 and gradients <= 1e-9 relative
(summation order only); mixed forces max_rel <= 1e-5 and mixed gradients
<= 1e-6 relative to the FP64 gradient.  The device FP64 gradient is also
checked against central differences (h = 1e-6) of the device FP64 loss."""
import numpy as np
import pytest

from oracle import fitref as FR
from gpu_helpers import force_errors

pytestmark = pytest.mark.gpu

from lammps_amd import batch as B  # noqa: E402
from lammps_amd import workloads as W  # noqa: E402

KA = W.KA_PAIRS


def ka_tables(pairs=KA):
    nt1 = 3
    e, s, c = np.zeros((nt1, nt1)), np.zeros((nt1, nt1)), np.zeros((nt1, nt1))
    for (a, b), (ee, ss, cc) in pairs.items():
        for i, j in ((a, b), (b, a)):
            e[i, j], s[i, j], c[i, j] = ee, ss, cc
    return e, s, c


def ka_batch_inputs(nrep=3, nside=10, seed=1):
    rng = np.random.default_rng(seed)
    xs, ts = [], []
    x0, t0, L = W.ka_initial(nside=nside, nb=int(0.2 * nside ** 3))
    for r in range(nrep):
        xs.append(x0 + rng.normal(scale=0.06, size=x0.shape))
        ts.append(t0)
    n = len(t0)
    return [n] * nrep, [[0, 0, 0]] * nrep, [[L, L, L]] * nrep, [[1, 1, 1]] * nrep, np.concatenate(ts), np.concatenate(xs)


@pytest.fixture(scope="module")
def ka():
    natoms, lo, hi, per, t, x = ka_batch_inputs()
    ref = FR.Batch(natoms, lo, hi, per, 2, t, x)
    e, s, c = ka_tables()
    f_ref, en_ref = ref.lj_forces(e, s, c)
    G = np.random.default_rng(7).normal(size=x.shape)
    ge_ref, gs_ref = ref.lj_vjp(e, s, c, G)
    return dict(natoms=natoms, lo=lo, hi=hi, per=per, t=t, x=x, f=f_ref, e=en_ref, G=G, ge=ge_ref, gs=gs_ref)


def make_lj(ka, precision):
    b = B.Batch(ka["natoms"], ka["lo"], ka["hi"], ka["per"], 2, ka["t"])
    b.set_positions(ka["x"])
    b.precision(precision)
    b.lj_init(*ka_tables())
    return b


def rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


def test_lj_batch_forces_fp64_and_mixed(ka):
    for prec, tol in ((B.FP64, 1e-11), (B.MIXED, 1e-5)):
        b = make_lj(ka, prec)
        f, e = b.lj_forces()
        mx, _ = force_errors(f, ka["f"])
        assert mx <= tol, (prec, mx)
        assert np.max(np.abs(e - ka["e"]) / np.abs(ka["e"])) <= (1e-12 if prec == B.FP64 else 1e-6)
        b.close()


def test_lj_batch_gradient_fp64_and_mixed(ka):
    for prec, tol in ((B.FP64, 1e-9), (B.MIXED, 1e-6)):
        b = make_lj(ka, prec)
        ge, gs = b.lj_vjp(ka["G"])
        for g, gr in ((ge, ka["ge"]), (gs, ka["gs"])):
            for a, c in ((1, 1), (1, 2), (2, 2)):
                assert abs(g[a, c] - gr[a, c]) <= tol * abs(gr[a, c]), (prec, a, c, g[a, c], gr[a, c])
        b.close()


def test_lj_batch_gradient_matches_device_finite_differences(ka):
    b = make_lj(ka, B.FP64)
    ge, gs = b.lj_vjp(ka["G"])
    e0, s0, c0 = ka_tables()
    for which, g in ((0, ge), (1, gs)):
        for a, c in ((1, 1), (1, 2), (2, 2)):
            vals = []
            base = (e0, s0)[which][a, c]
            h = 1e-6 * base
            for sgn in (1, -1):
                tabs = [e0.copy(), s0.copy()]
                tabs[which][a, c] += sgn * h
                tabs[which][c, a] = tabs[which][a, c]
                b.lj_init(tabs[0], tabs[1], c0)
                vals.append(np.sum(ka["G"] * b.lj_forces(energy=False)[0]))
            fd = (vals[0] - vals[1]) / (2 * h)
            assert abs(g[a, c] - fd) <= 1e-6 * abs(fd), (which, a, c, g[a, c], fd)
    b.close()


def test_autotuned_launch_gives_the_same_results(ka):
    b = make_lj(ka, B.FP64)
    f0, _ = b.lj_forces()
    ge0, gs0 = b.lj_vjp(ka["G"])
    b.autotune(True)
    f1, _ = b.lj_forces()
    ge1, gs1 = b.lj_vjp(ka["G"])
    assert force_errors(f1, f0)[0] <= 1e-12
    assert rel(ge1[1:, 1:], ge0[1:, 1:]) <= 1e-12 and rel(gs1[1:, 1:], gs0[1:, 1:]) <= 1e-12
    for kind in (B.BK_LJ, B.BK_LJ_VJP):
        sh = b.get_launch(kind)
        assert sh["tpa"] in (2, 4, 8, 16) and sh["block"] in (128, 256, 512)
    # explicit shapes, including a tiny grid that loops over many tiles
    for tpa, block, grid in ((1, 64, 1), (32, 1024, 0), (4, 128, 3)):
        b.set_launch(B.BK_LJ, block, tpa, grid)
        b.set_launch(B.BK_LJ_VJP, block, tpa, grid)
        assert force_errors(b.lj_forces()[0], f0)[0] <= 1e-12
        ge2, _ = b.lj_vjp(ka["G"])
        assert rel(ge2[1:, 1:], ge0[1:, 1:]) <= 1e-12
    b.close()


@pytest.fixture(scope="module")
def eam():
    pot = W.synthetic_knots(64)
    xs = [W.fcc_cluster(n) for n in (200, 431, 1000)]
    rng = np.random.default_rng(3)
    xs = [x + rng.normal(scale=0.12, size=x.shape) for x in xs]
    lo = [x.min(0) - 2.0 for x in xs]
    hi = [x.max(0) + 2.0 for x in xs]
    # plus a periodic crystal replica
    a = 3.615
    ncell = 4
    basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    g = np.stack(np.meshgrid(*(np.arange(ncell),) * 3, indexing="ij"), -1).reshape(-1, 3)
    xp = ((g[:, None, ::-1] + basis[None]) * a).reshape(-1, 3) + rng.normal(scale=0.1, size=(4 * ncell ** 3, 3))
    L = ncell * a
    xs.append(xp)
    lo.append([0, 0, 0])
    hi.append([L, L, L])
    per = [[0, 0, 0]] * 3 + [[1, 1, 1]]
    natoms = [len(x) for x in xs]
    x = np.concatenate(xs)
    ref = FR.Batch(natoms, lo, hi, per, 1, np.ones(len(x)), x)
    ref.eam_set(pot["drho"], pot["dr"], pot["cut"], pot["frho"], pot["rhor"], pot["z2r"])
    f, e, rho, fp = ref.eam_forces()
    G = np.random.default_rng(11).normal(size=x.shape)
    g = ref.eam_vjp(G)
    return dict(pot=pot, natoms=natoms, lo=lo, hi=hi, per=per, x=x, f=f, e=e, rho=rho, fp=fp, G=G, g=g)


def make_eam(d, precision):
    b = B.Batch(d["natoms"], d["lo"], d["hi"], d["per"], 1, np.ones(len(d["x"]), np.int32))
    b.set_positions(d["x"])
    b.precision(precision)
    p = d["pot"]
    b.eam_init(p["drho"], p["dr"], p["cut"], p["frho"], p["rhor"], p["z2r"])
    return b


def test_eam_batch_forces_fp64_and_mixed(eam):
    for prec, tol in ((B.FP64, 1e-11), (B.MIXED, 1e-5)):
        b = make_eam(eam, prec)
        f, e, rho, fp = b.eam_forces(rho_fp=True)
        assert force_errors(f, eam["f"])[0] <= tol, prec
        assert np.max(np.abs(e - eam["e"]) / np.abs(eam["e"])) <= (1e-12 if prec == B.FP64 else 1e-6)
        assert rel(rho, eam["rho"]) <= (1e-12 if prec == B.FP64 else 1e-6)
        b.close()


def test_eam_batch_knot_gradient_fp64_and_mixed(eam):
    for prec, tol in ((B.FP64, 1e-9), (B.MIXED, 1e-6)):
        b = make_eam(eam, prec)
        b.eam_forces()
        g = b.eam_vjp(eam["G"])
        for gd, gr in zip(g, eam["g"]):
            assert np.max(np.abs(gd - gr)) <= tol * np.max(np.abs(gr)), (prec, np.max(np.abs(gd - gr)))
        # a vjp without a preceding forward on these tables recomputes rho/fp
        b2 = make_eam(eam, prec)
        g2 = b2.eam_vjp(eam["G"])
        for gd, gr in zip(g2, eam["g"]):
            assert np.max(np.abs(gd - gr)) <= tol * np.max(np.abs(gr))
        b.close()
        b2.close()


def test_eam_batch_gradient_matches_device_finite_differences(eam):
    b = make_eam(eam, B.FP64)
    g = b.eam_vjp(eam["G"])
    p = eam["pot"]
    knots = [p["frho"], p["rhor"], p["z2r"]]
    rng = np.random.default_rng(2)
    for which in range(3):
        nz = np.nonzero(np.abs(g[which]) > 1e-3 * np.max(np.abs(g[which])))[0]
        for k in rng.choice(nz, size=min(8, len(nz)), replace=False):
            h = 1e-6 * max(abs(knots[which][k]), 1e-3)
            vals = []
            for sgn in (1, -1):
                kk = [a.copy() for a in knots]
                kk[which][k] += sgn * h
                b.eam_init(p["drho"], p["dr"], p["cut"], *kk)
                vals.append(np.sum(eam["G"] * b.eam_forces(energy=False)[0]))
            fd = (vals[0] - vals[1]) / (2 * h)
            assert abs(g[which][k] - fd) <= 1e-6 * np.max(np.abs(g[which])), (which, k, g[which][k], fd)
    b.close()


def test_torch_autograd_functions_match_the_adjoint(ka, eam):
    import torch

    from lammps_amd import fit

    dev = torch.device("cuda", 0)
    eps, sig, cut = W.ka_pair_vectors()
    fm = fit.LJForceMatch(ka["natoms"], ka["lo"], ka["hi"], ka["per"], 2, ka["t"], ka["x"], cut, precision=B.FP64)
    e_t = torch.tensor(eps, dtype=torch.float64, requires_grad=True)
    s_t = torch.tensor(sig, dtype=torch.float64, requires_grad=True)
    F = fm(e_t, s_t)
    assert F.is_cuda and F.shape == (len(ka["t"]), 3)
    assert force_errors(F.detach().cpu().numpy(), ka["f"])[0] <= 1e-11
    G = torch.tensor(ka["G"], device=dev)
    (F * G).sum().backward()
    for got, ref in ((e_t.grad.numpy(), ka["ge"]), (s_t.grad.numpy(), ka["gs"])):
        for v, (a, c) in zip(got, ((1, 1), (1, 2), (2, 2))):
            assert abs(v - ref[a, c]) <= 1e-9 * abs(ref[a, c])
    p = eam["pot"]
    em = fit.EAMForceMatch(eam["natoms"], eam["lo"], eam["hi"], eam["per"], eam["x"], p["drho"], p["dr"], p["cut"],
                           precision=B.FP64)
    kn = [torch.tensor(p[k], dtype=torch.float64, requires_grad=True) for k in ("frho", "rhor", "z2r")]
    F2 = em(*kn)
    (F2 * torch.tensor(eam["G"], device=dev)).sum().backward()
    for t, ref in zip(kn, eam["g"]):
        assert np.max(np.abs(t.grad.numpy() - ref)) <= 1e-9 * np.max(np.abs(ref))
    fm.batch.close()
    em.batch.close()


def test_neighbour_counts_match_brute_force_small_boxes():
    # periodic box of 2.1 cutoffs with few bins per dimension, and a cluster
    rng = np.random.default_rng(5)
    L = 2.1 * 2.5
    x1 = rng.uniform(0, L, size=(60, 3))
    x2 = rng.uniform(0, 6.0, size=(40, 3))
    x = np.concatenate([x1, x2])
    t = np.ones(100, np.int32)
    b = B.Batch([60, 40], [[0, 0, 0], [0, 0, 0]], [[L, L, L], [6, 6, 6]], [[1, 1, 1], [0, 0, 0]], 1, t)
    b.set_positions(x)
    one = np.ones((2, 2))
    b.lj_init(one, one * 0.5, one * 2.5)
    total, _ = b.neigh_stats()
    cnt = 0
    for i in range(60):
        d = x1 - x1[i]
        d -= L * np.round(d / L)
        r2 = np.sum(d * d, 1)
        cnt += int(np.sum(r2 < 2.5 ** 2)) - 1
    for i in range(40):
        r2 = np.sum((x2 - x2[i]) ** 2, 1)
        cnt += int(np.sum(r2 < 2.5 ** 2)) - 1
    assert total == cnt
    b.close()


@pytest.mark.parametrize("density", [0.9, 7.0])
@pytest.mark.parametrize("side", [(2.1, 2.3, 2.2), (2.6, 5.3, 3.1), (9.7, 2.6, 2.6)])
def test_neighbour_counts_match_brute_force(side, density):
    """Boxes of four bins a side (FP64 candidates) and of more (fixed-point
    candidates), a free cluster beside each, rows of more candidates than one
    window of the build holds (density 7: about 460 neighbours per atom)."""
    rng = np.random.default_rng(8)
    L = 2.5 * np.array(side)
    n1 = int(density * np.prod(L))
    x1 = rng.uniform(0, 1, size=(n1, 3)) * L
    x2 = rng.uniform(0, 1, size=(n1 // 2 + 1, 3)) * L
    b = B.Batch([n1, len(x2)], [[0, 0, 0]] * 2, [L, L], [[1, 1, 1], [0, 0, 0]], 1, np.ones(n1 + len(x2), np.int32))
    b.set_positions(np.concatenate([x1, x2]))
    one = np.ones((2, 2))
    b.lj_init(one, one * 0.5, one * 2.5)
    total, most = b.neigh_stats()
    counts = []
    for x, periodic in ((x1, True), (x2, False)):
        for i in range(len(x)):
            d = x - x[i]
            if periodic:
                d -= L * np.round(d / L)
            counts.append(int(np.sum(np.sum(d * d, 1) < 2.5 ** 2)) - 1)
    assert total == sum(counts) and most == max(counts)
    b.close()


@pytest.mark.parametrize("ntypes", [1, 3, 8])
def test_lj_gradient_for_other_type_counts(ntypes):
    """One type, and the general kernel of three or more (two: the
    Kob-Andersen tests): forces and gradients equal the oracle's, a periodic
    box and a free one, a different cutoff for every type pair."""
    rng = np.random.default_rng(ntypes)
    L, n = 9.3, (701, 307)
    grid = np.stack(np.meshgrid(*(np.arange(9),) * 3, indexing="ij"), -1).reshape(-1, 3) * (L / 9) + 0.2
    x = np.concatenate([grid[rng.permutation(len(grid))[:m]] + rng.uniform(-0.15, 0.15, (m, 3)) for m in n])
    t = rng.integers(1, ntypes + 1, len(x)).astype(np.int32)
    e, s, c = (np.zeros((ntypes + 1, ntypes + 1)) for _ in range(3))
    for i in range(1, ntypes + 1):
        for j in range(i, ntypes + 1):
            e[i, j] = e[j, i] = rng.uniform(0.5, 1.5)
            s[i, j] = s[j, i] = rng.uniform(0.8, 1.0)
            c[i, j] = c[j, i] = rng.uniform(2.0, 2.5)
    geo = (list(n), [[0, 0, 0], [0, 0, 0]], [[L, L, L]] * 2, [[1, 1, 1], [0, 0, 0]], ntypes, t)
    x = np.clip(x, 0.0, L - 1e-9)
    ref = FR.Batch(*geo, x)
    G = rng.normal(size=x.shape)
    ge_ref, gs_ref = ref.lj_vjp(e, s, c, G)
    b = B.Batch(*geo)
    b.set_positions(x)
    b.lj_init(e, s, c)
    assert force_errors(b.lj_forces()[0], ref.lj_forces(e, s, c)[0])[0] <= 1e-11
    ge, gs = b.lj_vjp(G)
    assert rel(ge, ge_ref) <= 1e-9 and rel(gs, gs_ref) <= 1e-9
    b.close()


@pytest.mark.parametrize("nknots", [16, 300, 511, 512, 660])
def test_eam_table_sizes(nknots):
    """Tables in LDS and beyond it (the FP64 force pass to 511 knots, several
    adjoint accumulator sets only below ~90): forces and knot gradients equal
    the oracle's."""
    pot = W.synthetic_knots(nknots)
    rng = np.random.default_rng(nknots)
    xs = [q + rng.normal(scale=0.1, size=q.shape) for q in (W.fcc_cluster(331), W.fcc_cluster(120))]
    x = np.concatenate(xs)
    geo = ([len(q) for q in xs], [q.min(0) - 2.0 for q in xs], [q.max(0) + 2.0 for q in xs], [[0, 0, 0]] * 2, 1,
           np.ones(len(x), np.int32))
    ref = FR.Batch(*geo, x)
    ref.eam_set(pot["drho"], pot["dr"], pot["cut"], pot["frho"], pot["rhor"], pot["z2r"])
    G = rng.normal(size=x.shape)
    g_ref = ref.eam_vjp(G)
    f_ref = ref.eam_forces()[0]
    for prec, tol in ((B.FP64, 1e-11), (B.MIXED, 1e-5)):
        b = B.Batch(*geo)
        b.set_positions(x)
        b.precision(prec)
        b.eam_init(pot["drho"], pot["dr"], pot["cut"], pot["frho"], pot["rhor"], pot["z2r"])
        assert force_errors(b.eam_forces()[0], f_ref)[0] <= tol
        for gd, gr in zip(b.eam_vjp(G), g_ref):
            assert np.max(np.abs(gd - gr)) <= 1e-9 * np.max(np.abs(gr))
        b.close()


@pytest.mark.parametrize("nrep,nside", [(2, 17), (3, 15), (10, 17), (11, 17)])
def test_default_batch_launch_shapes_agree_with_a_fixed_one(nrep, nside):
    """Batches on both sides of the sizes (10,000 and 50,000 atoms) where the
    default launch shape changes, against workgroups of 256 at 8 lanes."""
    natoms, lo, hi, per, t, x = ka_batch_inputs(nrep, nside)
    b = B.Batch(natoms, lo, hi, per, 2, t)
    b.set_positions(x)
    b.lj_init(*ka_tables())
    G = np.random.default_rng(2).normal(size=x.shape)
    f0, (ge0, gs0) = b.lj_forces()[0], b.lj_vjp(G)
    for kind in (B.BK_LJ, B.BK_LJ_VJP):
        b.set_launch(kind, 256, 8, 0)
    f1, (ge1, gs1) = b.lj_forces()[0], b.lj_vjp(G)
    assert force_errors(f0, f1)[0] <= 1e-12
    assert rel(ge0, ge1) <= 1e-12 and rel(gs0, gs1) <= 1e-12
    b.close()


@pytest.mark.parametrize("far", [5.0, 1e9, 1e30, np.inf, -1e9, -np.inf, np.nan])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_atom_far_outside_a_closed_box_is_reported(d, far):
    """An atom outside its replica's box in a non-periodic dimension is an
    error, however far outside it lies; the batch works on afterwards."""
    rng = np.random.default_rng(3)
    x = rng.uniform(0.2, 19.8, size=(600, 3))
    b = B.Batch([400, 200], [[0, 0, 0]] * 2, [[20.0, 20.0, 20.0]] * 2, [[0, 0, 0]] * 2, 1, np.ones(600, np.int32))
    one = np.ones((2, 2))
    b.lj_init(one, one * 0.1, one * 2.5)
    bad = x.copy()
    bad[399, d] = 20.0 + far if far > 0 or far != far else far
    b.set_positions(bad)
    with pytest.raises(Exception, match="outside its replica's box"):
        b.neigh_stats()
    b.set_positions(x)
    total, _ = b.neigh_stats()
    want = sum(int(np.sum(np.sum((q[:, None] - q[None]) ** 2, -1) < 6.25)) - len(q) for q in (x[:400], x[400:]))
    assert total == want
    b.close()


@pytest.mark.parametrize("tpa,nknots", [(4, 64), (16, 64), (4, 660), (16, 660)])
def test_coincident_eam_atoms_have_the_density_of_zero_separation(tpa, nknots):
    """Two atoms of a cluster in one place (FP64, tables in LDS and not):
    densities and the forces on all other atoms are the oracle's."""
    pot = W.synthetic_knots(nknots)
    rng = np.random.default_rng(nknots)
    x = W.fcc_cluster(331) + rng.normal(scale=0.1, size=(331, 3))
    x[200] = x[17]
    geo = ([331], [x.min(0) - 2.0], [x.max(0) + 2.0], [[0, 0, 0]], 1, np.ones(331, np.int32))
    ref = FR.Batch(*geo, x)
    ref.eam_set(pot["drho"], pot["dr"], pot["cut"], pot["frho"], pot["rhor"], pot["z2r"])
    f_ref, _, rho_ref, fp_ref = ref.eam_forces()
    b = B.Batch(*geo)
    b.set_positions(x)
    b.eam_init(pot["drho"], pot["dr"], pot["cut"], pot["frho"], pot["rhor"], pot["z2r"])
    for kind in (B.BK_EAM_RHO, B.BK_EAM_FORCE):
        b.set_launch(kind, 256, tpa, 0)
    f, _, rho, fp = b.eam_forces(rho_fp=True)
    assert np.isfinite(rho_ref).all()
    np.testing.assert_allclose(rho, rho_ref, rtol=1e-11)
    np.testing.assert_allclose(fp, fp_ref, rtol=0, atol=1e-10 * np.abs(fp_ref).max())
    rest = np.setdiff1d(np.arange(331), [17, 200])
    assert force_errors(f[rest], f_ref[rest])[0] <= 1e-11
    b.close()


def test_build_kind_reports_the_shape_it_runs():
    """The list build takes its own launch shape whatever is set for it."""
    natoms, lo, hi, per, t, x = ka_batch_inputs(2, 8)
    b = B.Batch(natoms, lo, hi, per, 2, t)
    b.set_positions(x)
    b.lj_init(*ka_tables())
    shape = b.get_launch(B.BK_BUILD)
    assert shape["block"] == 256 and shape["tpa"] == 32 and shape["grid"] == 128
    b.set_launch(B.BK_BUILD, 512, 4, 7)
    assert b.get_launch(B.BK_BUILD) == shape
    b.autotune(True)
    b.lj_forces()
    assert b.get_launch(B.BK_BUILD) == shape
    b.close()


def boundary_pairs(L, cut, want=240):
    """Two-atom boxes whose atoms lie within a few ulps of `cut` apart through
    a periodic face: positions [m, 2, 3], only pairs where x_i - (x_j + L),
    x_j - (x_i - L) and the nearest image of x_i - x_j do not all decide alike."""
    rng = np.random.default_rng(17)
    out = []
    while len(out) < want:
        d = int(rng.integers(3))
        x = np.tile(rng.uniform(1.0, 9.0, 3), (2, 1))
        lowside = rng.uniform(0.0, 1.0)
        high = L[d] + lowside - cut
        x[0, d], x[1, d] = high + int(rng.integers(-3, 4)) * np.spacing(high), lowside
        i, j = (0, 1) if rng.random() < 0.5 else (1, 0)
        a = x[0, d] - (x[1, d] + L[d])
        b = x[1, d] - (x[0, d] - L[d])
        c = (x[0, d] - x[1, d]) - L[d]
        if len({q * q < cut * cut for q in (a, b, c)}) > 1:
            out.append(x[[i, j]])
    return np.array(out)


@pytest.mark.parametrize("skin", [0.0, 0.3])
@pytest.mark.parametrize("tpa", [4, 16])
def test_pairs_at_the_cutoff_through_a_periodic_face(skin, tpa):
    """A pair is decided by the FP64 separation from the neighbour's image,
    x_i - (x_j + shift), in each row by itself: forces, energies and parameter
    gradients of pairs on the cutoff are the oracle's, in both precisions."""
    L = np.array([11.3, 12.7, 13.9])
    one = np.ones((2, 2))
    rng = np.random.default_rng(1)
    for style, cut in (("lj", 2.5), ("eam", 4.95)):
        x = boundary_pairs(L, cut)
        m = len(x)
        x = x.reshape(-1, 3)
        geo = ([2] * m, [[0, 0, 0]] * m, [L] * m, [[1, 1, 1]] * m, 1, np.ones(2 * m, np.int32))
        ref = FR.Batch(*geo, x)
        G = rng.normal(size=x.shape)
        b = B.Batch(*geo)
        b.set_positions(x)
        b.skin(skin)
        for kind in range(1, 7):
            b.set_launch(kind, 256, tpa, 0)
        if style == "lj":
            args = (one, one, one * cut)
            f_ref, e_ref = ref.lj_forces(*args)
            g_ref = ref.lj_vjp(*args, G)
            b.lj_init(*args)
        else:
            pot = W.synthetic_knots(64)
            args = (pot["drho"], pot["dr"], cut, pot["frho"], pot["rhor"], pot["z2r"])
            ref.eam_set(*args)
            f_ref, e_ref = ref.eam_forces()[:2]
            g_ref = ref.eam_vjp(G)
            b.eam_init(*args)
        for prec, ftol, etol in ((B.FP64, 1e-11, 1e-12), (B.MIXED, 1e-5, 1e-5)):
            b.precision(prec)
            f, e = b.lj_forces() if style == "lj" else b.eam_forces()
            assert force_errors(f, f_ref)[0] <= ftol
            assert np.max(np.abs(e - e_ref)) <= etol * np.max(np.abs(e_ref))
            for gd, gr in zip(b.lj_vjp(G) if style == "lj" else b.eam_vjp(G), g_ref):
                assert np.max(np.abs(gd - gr)) <= 1e-9 * np.max(np.abs(gr))
        b.close()


@pytest.mark.parametrize("tpa", [1, 4, 64])
def test_pairs_at_the_cutoff_in_long_rows(tpa):
    """The same among other neighbours, in rows of up to 40 trips of one lane:
    a jittered lattice of about 130 neighbours per atom with such pairs put in."""
    rng = np.random.default_rng(6)
    for style, cut, a, sigma in (("lj", 2.5, 0.78, 0.5), ("eam", 4.95, 1.56, None)):
        L = np.round(np.array([15, 16, 18]) * a, 2)
        ends = boundary_pairs(L, cut, 60)
        n = np.floor(L / a).astype(int)
        grid = np.stack(np.meshgrid(*[np.arange(q) for q in n], indexing="ij"), -1).reshape(-1, 3) * (L / n)
        grid = np.mod(grid + rng.uniform(-0.1 * a, 0.1 * a, grid.shape), L)
        taken = []
        for pair in ends:  # pairs whose atoms keep apart
            d = (pair[:, None] - np.array(taken).reshape(-1, 3)[None])
            d -= L * np.round(d / L)
            if not len(taken) or np.min(np.sum(d * d, -1)) > a * a:
                taken.extend(pair)
        taken = np.array(taken)
        d = grid[:, None] - taken[None]
        d -= L * np.round(d / L)
        x = np.concatenate([grid[np.min(np.sum(d * d, -1), 1) > (0.7 * a) ** 2], taken])
        x = x[rng.permutation(len(x))]
        assert len(taken) >= 20
        geo = ([len(x)], [[0, 0, 0]], [L], [[1, 1, 1]], 1, np.ones(len(x), np.int32))
        ref = FR.Batch(*geo, x)
        G = rng.normal(size=x.shape)
        b = B.Batch(*geo)
        b.set_positions(x)
        b.skin(0.05 * cut)
        for kind in range(1, 7):
            b.set_launch(kind, 256, tpa, 0)
        if style == "lj":
            one = np.ones((2, 2))
            args = (one, one * sigma, one * cut)
            f_ref, g_ref = ref.lj_forces(*args)[0], ref.lj_vjp(*args, G)
            b.lj_init(*args)
            f, g = b.lj_forces()[0], b.lj_vjp(G)
        else:
            pot = W.synthetic_knots(64)
            args = (pot["drho"], pot["dr"], cut, pot["frho"], pot["rhor"], pot["z2r"])
            ref.eam_set(*args)
            f_ref, g_ref = ref.eam_forces()[0], ref.eam_vjp(G)
            b.eam_init(*args)
            f, g = b.eam_forces()[0], b.eam_vjp(G)
        assert b.neigh_stats()[1] > (128 if tpa == 1 else 4)
        assert np.max(np.abs(f - f_ref)) <= 1e-11 * max(1.0, np.sqrt(np.mean(f_ref ** 2)))
        for gd, gr in zip(g, g_ref):
            assert np.max(np.abs(gd - gr)) <= 1e-9 * np.max(np.abs(gr))
        b.close()


@pytest.mark.parametrize("shell", [(1, 2, 0), (1, 1, 1), (2, 1, 1), (2, 2, 1)])
@pytest.mark.parametrize("skin", [0.0, 0.2])
def test_lattice_shell_at_the_cutoff(shell, skin):
    """A perfect simple-cubic lattice whose spacing is no exact fraction, the
    cutoff on one of its shells: each of thousands of ties is decided as the
    oracle's FP64 rounding of every product and sum decides it."""
    a = 1.1
    n = 8
    grid = np.stack(np.meshgrid(*(np.arange(n),) * 3, indexing="ij"), -1).reshape(-1, 3) * a
    cut = float(np.sqrt(np.sum((np.array(shell) * a) ** 2)))
    L = n * a
    geo = ([len(grid)] * 2, [[0, 0, 0]] * 2, [[L, L, L]] * 2, [[1, 1, 1], [0, 0, 0]], 1, np.ones(2 * len(grid), np.int32))
    x = np.concatenate([grid, grid])
    one = np.ones((2, 2))
    args = (one, one, one * cut)
    ref = FR.Batch(*geo, x)
    G = np.random.default_rng(3).normal(size=x.shape)
    f_ref, e_ref = ref.lj_forces(*args)
    g_ref = ref.lj_vjp(*args, G)
    b = B.Batch(*geo)
    b.set_positions(x)
    b.skin(skin)
    b.lj_init(*args)
    for prec, ftol in ((B.FP64, 1e-11), (B.MIXED, 1e-5)):
        b.precision(prec)
        f, e = b.lj_forces()
        scale = 24.0 * (2.0 / a ** 13 - 1.0 / a ** 7)  # a nearest pair's force: the lattice's cancel
        assert np.max(np.abs(f - f_ref)) <= ftol * scale
        assert np.max(np.abs(e - e_ref)) <= (1e-12 if prec == B.FP64 else 1e-5) * np.max(np.abs(e_ref))
        for gd, gr in zip(b.lj_vjp(G), g_ref):
            assert np.max(np.abs(gd - gr)) <= 1e-9 * np.max(np.abs(gr))
    b.close()


@pytest.mark.parametrize("bad", [np.nan, -np.nan])
@pytest.mark.parametrize("prec", [B.FP64, B.MIXED])
def test_atom_without_a_place_touches_no_other(prec, bad):
    """A coordinate that is not a number in a periodic box: the atom has no
    neighbours, whatever the fixed-point mirror makes of it, and all other
    atoms have the forces and gradients of the batch without it."""
    natoms, lo, hi, per, t, x = ka_batch_inputs(2, 9)
    n = natoms[0]
    lost = int(np.argmin(np.sum(x[:n] ** 2, 1)))  # beside the box's corner, among neighbours
    keep = np.delete(np.arange(2 * n), lost)
    G = np.random.default_rng(2).normal(size=x.shape)
    tab = ka_tables()
    want = B.Batch([n - 1, n], lo, hi, per, 2, t[keep])
    want.set_positions(x[keep])
    got = B.Batch(natoms, lo, hi, per, 2, t)
    broken = x.copy()
    broken[lost, 1] = np.copysign(np.nan, 1.0 if not np.signbit(bad) else -1.0)
    got.set_positions(broken)
    out = []
    for b, g in ((want, G[keep]), (got, G)):
        b.precision(prec)
        b.lj_init(*tab)
        out.append((b.neigh_stats()[0], b.lj_forces(), b.lj_vjp(g)))
        b.close()
    assert out[0][0] == out[1][0]
    assert not out[1][1][0][lost].any()
    assert force_errors(out[1][1][0][keep], out[0][1][0])[0] <= 1e-12
    assert np.max(np.abs(out[0][1][1] - out[1][1][1])) <= 1e-12 * np.max(np.abs(out[0][1][1]))
    for a, c in zip(out[0][2], out[1][2]):
        assert rel(c, a) <= 1e-12
