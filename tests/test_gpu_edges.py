"""GPU edge cases of the C ABI: tiny, empty and ragged systems, closed forms,
list capacity regrowth, and the errors the reference raises for them.

Bars (stated here, in the test):
  * closed forms (lj/cut dimer, pair_lj_cut.cpp:68-141): FP64 rel <= 1e-13,
    mixed rel <= 1e-6;
  * ragged random systems against the FP64 oracle: FP64 max_rel <= 1e-11,
    mixed <= 1e-5, pair sets identical;
  * error paths: the status code and the reference's message, no crash.
"""
import numpy as np
import pytest

from gpu_helpers import force_errors
from oracle import mdref as M

pytestmark = pytest.mark.gpu

MASS = np.array([0.0, 1.0])


def lj_context(lo, hi, periodic, x, prec, skin=0.3, one=2000, shift=False):
    from lammps_amd import mdx
    ctx = mdx.Context(0)
    ctx.set_box(lo, hi, periodic)
    ctx.set_atoms(x, np.ones(len(x), dtype=np.int32), MASS, tags=np.arange(1, len(x) + 1))
    ctx.pair_lj_from_coeffs(1, {(1, 1): (1.0, 1.0, 2.5)}, shift=shift)
    ctx.precision(prec)
    ctx.neigh_modify(skin, one=one)
    return ctx


def lj_dimer(r):
    """force on atom 0 along +x (atom 1 at +r) and the pair energy, 12-6 LJ"""
    f = 24.0 * (2.0 / r ** 13 - 1.0 / r ** 7)
    return -f, 4.0 * (r ** -12 - r ** -6)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("where", ["inside", "across_boundary", "closed_box"])
def test_lj_dimer_matches_closed_form(prec, where):
    from lammps_amd import mdx
    r0 = 1.05
    L = 10.0
    if where == "inside":
        x = np.array([[4.0, 5.0, 5.0], [4.0 + r0, 5.0, 5.0]])
        per = (1, 1, 1)
    elif where == "across_boundary":  # the pair only exists through the periodic image
        x = np.array([[L - 0.4, 5.0, 5.0], [r0 - 0.4, 5.0, 5.0]])
        per = (1, 1, 1)
    else:
        x = np.array([[4.0, 5.0, 5.0], [4.0 + r0, 5.0, 5.0]])
        per = (0, 0, 0)
    # the separation of these doubles as the reference forms it: the ghost
    # image x_j + L, then x_i - ghost (atom_vec_atomic.cpp:290-297)
    ghost = x[1, 0] + L if where == "across_boundary" else x[1, 0]
    r = ghost - x[0, 0]
    p = mdx.FP64 if prec == "fp64" else mdx.MIXED
    ctx = lj_context((0, 0, 0), (L, L, L), per, x, p)
    out = ctx.compute(1, 1)
    fx, e = lj_dimer(r)
    tol = 1e-13 if prec == "fp64" else 1e-6
    assert abs(out["f"][0, 0] - fx) <= tol * abs(fx)
    assert abs(out["f"][1, 0] + fx) <= tol * abs(fx)
    assert np.all(np.abs(out["f"][:, 1:]) <= tol * abs(fx))
    assert abs(out["eng"] - e) <= tol * abs(e)
    # virial xx of one pair: del_x * f_x (pair.cpp:769-855)
    assert abs(out["virial"][0] - r * (-fx)) <= tol * abs(r * fx)
    assert ctx.stats()["total_neighbors"] == 2
    ctx.close()


def test_single_atom_and_empty_system():
    from lammps_amd import mdx
    ctx = lj_context((0, 0, 0), (10, 10, 10), (1, 1, 1), np.array([[1.0, 2.0, 3.0]]), mdx.FP64)
    out = ctx.compute(1, 1)
    assert np.all(out["f"] == 0.0) and out["eng"] == 0.0 and np.all(out["virial"] == 0.0)
    assert ctx.stats()["total_neighbors"] == 0
    ctx.close()
    ctx = lj_context((0, 0, 0), (10, 10, 10), (1, 1, 1), np.zeros((0, 3)), mdx.MIXED)
    out = ctx.compute(1, 1)
    assert out["f"].shape == (0, 3) and out["eng"] == 0.0 and np.all(out["virial"] == 0.0)
    ctx.setup()
    ctx.run(5, 0.005, 1.0, 5)
    ctx.close()


def random_gas(n, L, dmin, seed):
    """n points in [0, L)^3 with minimum-image separation >= dmin"""
    rng = np.random.default_rng(seed)
    pts = np.zeros((0, 3))
    while len(pts) < n:
        p = rng.uniform(0.0, L, 3)
        d = (pts - p + L / 2) % L - L / 2
        if len(pts) == 0 or np.min(np.einsum("ij,ij->i", d, d)) >= dmin * dmin:
            pts = np.vstack([pts, p])
    return pts


@pytest.mark.parametrize("n", [37, 300, 1025])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_ragged_random_systems_match_the_oracle(n, prec):
    """atom counts that fill no block or wavefront evenly"""
    from lammps_amd import mdx
    L = 8.0 if n < 300 else 11.0
    x = random_gas(n, L, 0.85, seed=n)
    t = np.ones(n, dtype=np.int32)
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), (L, L, L))
    ref.add_atoms(x, t)
    ref.mass(1, 1.0)
    ref.pair_lj(2.5)
    ref.pair_coeff(1, 1, 1.0, 1.0, 2.5)
    ref.neighbor(0.3)
    ref.setup()
    _, _, fref, _, _ = ref.state()
    eref, _ = ref.energy_virial()
    ctx = lj_context((0, 0, 0), (L, L, L), (1, 1, 1), x, mdx.FP64 if prec == "fp64" else mdx.MIXED)
    out = ctx.compute(1, 1)
    got = {(int(a), int(b)) for a, b in ctx.neigh_pairs()}
    assert got == {(min(a, b), max(a, b)) for a, b in ref.list_pairs()}
    mx, _ = force_errors(out["f"], fref)
    assert mx <= (1e-11 if prec == "fp64" else 1e-5)
    assert abs(out["eng"] - eref) <= (1e-11 if prec == "fp64" else 1e-6) * abs(eref)
    ctx.close()


def oracle_lj_pairs_forces(lo, hi, periodic, x):
    ref = M.Ref(M.LJ)
    ref.box(lo, hi, periodic)
    ref.add_atoms(x, np.ones(len(x), dtype=np.int32))
    ref.mass(1, 1.0)
    ref.pair_lj(2.5)
    ref.pair_coeff(1, 1, 1.0, 1.0, 2.5)
    ref.neighbor(0.3)
    ref.setup()
    return {(min(a, b), max(a, b)) for a, b in ref.list_pairs()}, ref.state()[2]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", ["four_bins", "thin_slab"])
def test_small_bin_grids_match_the_oracle(prec, shape):
    """Bin grids at the edges of the list build's layouts.  four_bins: a
    periodic box of 4 bins a side (just above twice the neighbour cutoff),
    where a stencil row of 5 bins wraps onto bins it already holds, the
    same atoms under two images.  thin_slab: a closed dimension thinner
    than half the cutoff (one bin, so a stencil of 7 planes), which takes
    the per-row build."""
    from lammps_amd import mdx
    if shape == "four_bins":
        L = 5.8
        x = random_gas(110, L, 0.9, seed=11)
        lo, hi, per = (0.0, 0.0, 0.0), (L, L, L), (1, 1, 1)
    else:
        rng = np.random.default_rng(12)
        pts = np.zeros((0, 3))
        while len(pts) < 90:
            p = rng.uniform((0.0, 0.0, 0.05), (10.0, 10.0, 0.95))
            d = pts - p
            d[:, :2] = (d[:, :2] + 5.0) % 10.0 - 5.0
            if len(pts) == 0 or np.min(np.einsum("ij,ij->i", d, d)) >= 0.81:
                pts = np.vstack([pts, p])
        x = pts
        lo, hi, per = (0.0, 0.0, 0.0), (10.0, 10.0, 1.0), (1, 1, 0)
    want, fref = oracle_lj_pairs_forces(lo, hi, per, x)
    ctx = lj_context(lo, hi, per, x, mdx.FP64 if prec == "fp64" else mdx.MIXED)
    out = ctx.compute(1, 1)
    got = {(int(a), int(b)) for a, b in ctx.neigh_pairs()}
    st = ctx.stats()
    ctx.close()
    assert shape != "thin_slab" or st["nbins"][2] == 1
    assert shape != "four_bins" or st["nbins"][0] == 4
    assert len(want) > 0 and got == want
    mx, _ = force_errors(out["f"], fref)
    assert mx <= (1e-11 if prec == "fp64" else 1e-5)


@pytest.mark.parametrize("nb", [(5, 5, 5), (15, 21, 13), (16, 16, 16), (43, 37, 5), (16, 16, 32), (25, 31, 21),
                                (16, 32, 32), (31, 33, 32), (32, 32, 32)])
def test_bin_counts_around_the_scan_lines(nb):
    """Grids whose counters (bins + 1) end just below, at and above the lines
    where the scan of the bin counters changes (4,096, 8,192, 16,384 and
    32,768 counters), and in between: the pairs are those of a search over
    all atoms."""
    from scipy.spatial import cKDTree
    from lammps_amd import mdx
    cut = 2.8  # 2.5 and the skin; two bins to the cutoff
    L = 0.5 * cut * np.array(nb) + 0.2
    x = np.random.default_rng(sum(nb)).uniform(0.0, 1.0, (3000, 3)) * L
    ctx = lj_context((0.0, 0.0, 0.0), tuple(L), (1, 1, 1), x, mdx.FP64)
    ctx.neigh_build()
    got = {(min(int(a), int(b)) - 1, max(int(a), int(b)) - 1) for a, b in ctx.neigh_pairs()}  # pairs of tags
    st = ctx.stats()
    ctx.close()
    assert tuple(st["nbins"]) == nb
    assert got == cKDTree(x, boxsize=L).query_pairs(cut)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_long_box_beyond_the_pruning_grid_matches_the_oracle(prec):
    """A periodic box 12,000 sigma long in x: more than 8192 bins in x, where
    the build skips its per-atom stencil pruning (its FP32 bin coordinates
    would lose the margins), and a fixed-point mirror too coarse for the
    cutoff band, so both precisions test FP64 candidates.  Clumps of atoms
    along x, one across the periodic face."""
    from lammps_amd import mdx
    Lx, Ly = 12000.0, 6.0
    rng = np.random.default_rng(21)
    pts = np.zeros((0, 3))
    for cx in (1.0, 3000.0, 7000.5, Lx - 1.5):
        while len(pts) < 40 * (1 + int(np.sum([cx > c for c in (1.0, 3000.0, 7000.5)]))):
            p = np.array([cx + rng.uniform(-2.5, 2.5), rng.uniform(0.0, Ly), rng.uniform(0.0, Ly)])
            p[0] %= Lx
            d = pts - p
            d[:, 0] = (d[:, 0] + Lx / 2) % Lx - Lx / 2
            d[:, 1:] = (d[:, 1:] + Ly / 2) % Ly - Ly / 2
            if len(pts) == 0 or np.min(np.einsum("ij,ij->i", d, d)) >= 0.81:
                pts = np.vstack([pts, p])
    lo, hi, per = (0.0, 0.0, 0.0), (Lx, Ly, Ly), (1, 1, 1)
    want, fref = oracle_lj_pairs_forces(lo, hi, per, pts)
    ctx = lj_context(lo, hi, per, pts, mdx.FP64 if prec == "fp64" else mdx.MIXED)
    out = ctx.compute(1, 1)
    got = {(int(a), int(b)) for a, b in ctx.neigh_pairs()}
    st = ctx.stats()
    ctx.close()
    assert st["nbins"][0] > 8192
    assert len(want) > 0 and got == want
    mx, _ = force_errors(out["f"], fref)
    assert mx <= (1e-11 if prec == "fp64" else 1e-5)


def test_list_capacity_regrows_for_a_dense_cluster():
    """A compact fcc droplet in a large periodic box: the first-guess row
    capacity comes from the mean density (far below the droplet's ~78
    neighbours), so the build must regrow it (the accelerator library's
    max_nbors resize) and still give the oracle's forces."""
    from lammps_amd import mdx
    a = (4.0 / 0.8442) ** (1.0 / 3.0)
    basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    g = np.stack(np.meshgrid(*(np.arange(5),) * 3, indexing="ij"), -1).reshape(-1, 3)
    x = ((g[:, None] + basis[None]) * a).reshape(-1, 3) + 10.0
    L = 40.0
    ctx = lj_context((0, 0, 0), (L, L, L), (1, 1, 1), x, mdx.FP64)
    out = ctx.compute(1, 1)
    st = ctx.stats()
    assert st["max_neighbors"] > 60 and st["capacity"] >= st["max_neighbors"]
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), (L, L, L))
    ref.add_atoms(x, np.ones(len(x), dtype=np.int32))
    ref.mass(1, 1.0)
    ref.pair_lj(2.5)
    ref.pair_coeff(1, 1, 1.0, 1.0, 2.5)
    ref.neighbor(0.3)
    ref.setup()
    mx, _ = force_errors(out["f"], ref.state()[2])
    assert mx <= 1e-11
    ctx.close()


def test_neighbor_overflow_is_reported():
    """neigh_modify one below the per-atom count: the reference's error
    (neigh_half_bin.cpp:414-415), as a status code, not a crash"""
    from lammps_amd import mdx
    a = (4.0 / 0.8442) ** (1.0 / 3.0)
    _, _, x = mdx.lattice("fcc", 0.8442, "lj", (0, 0, 0), (6, 6, 6))
    ctx = lj_context((0, 0, 0), (6 * a,) * 3, (1, 1, 1), x, mdx.MIXED, one=20)
    with pytest.raises(mdx.MdxError) as e:
        ctx.compute(1, 1)
    assert e.value.code == mdx.ERR_OVERFLOW and "boost neigh_modify one" in str(e.value)
    ctx.close()


def _crowded(ncrowd, seed):
    """A sparse periodic background plus `ncrowd` atoms inside one bin:
    box 20 sigma, neighbour cutoff 2.8, 14 bins of 1.4286 per dimension, the
    crowd uniform in [5.75, 6.9)^3 (bin 4 in each dimension)."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*(np.arange(10),) * 3, indexing="ij"), -1).reshape(-1, 3) * 2.0 + 0.5
    g = g[np.any(np.abs(g - 6.3) > 3.5, axis=1)]  # keep the background clear of the crowd
    return np.vstack([g, 5.75 + 1.15 * rng.random((ncrowd, 3))])


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_crowded_bin_gives_the_oracle_pair_set(prec):
    """400 atoms in one bin (each has >= 399 neighbours, one = 2000 allows
    them): the per-bin ranking of the counting sort runs over the whole bin
    and the list equals the oracle's half_bin_newton pair set."""
    from lammps_amd import mdx
    x = _crowded(400, 3)
    L = 20.0
    ctx = lj_context((0, 0, 0), (L, L, L), (1, 1, 1), x, mdx.FP64 if prec == "fp64" else mdx.MIXED)
    ctx.neigh_build()
    st = ctx.stats()
    assert st["max_neighbors"] >= 399
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), (L, L, L))
    ref.add_atoms(x, np.ones(len(x), dtype=np.int32))
    ref.mass(1, 1.0)
    ref.pair_lj(2.5)
    ref.pair_coeff(1, 1, 1.0, 1.0, 2.5)
    ref.neighbor(0.3)
    ref.setup()
    got = np.sort(np.array([min(a, b) << 32 | max(a, b) for a, b in ctx.neigh_pairs()], dtype=np.int64))
    want = np.sort(np.array([min(a, b) << 32 | max(a, b) for a, b in ref.list_pairs()], dtype=np.int64))
    assert np.array_equal(got, want)
    ctx.close()


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("n", [163839, 163840, 163841])
def test_list_on_both_sides_of_the_build_size_line_matches_the_oracle(n, fmt):
    """Around 163,840 atoms the build changes from 32 lanes per atom to one:
    two types, a closed y dimension, an odd last atom, FP64 and fixed-point
    candidates; the pair set equals the oracle's."""
    from lammps_amd import mdx
    cells = (35, 34, 35)
    rng = np.random.default_rng(5)
    lo, hi, x = mdx.lattice("fcc", 0.8442, "lj", (0, 0, 0), cells)
    x = x[rng.permutation(len(x))[:n]] + rng.uniform(-0.1, 0.1, (n, 3))
    lo, hi = np.asarray(lo).copy(), np.asarray(hi).copy()
    x[:, 0::2] = np.mod(x[:, 0::2], hi[0::2])
    lo[1], hi[1] = -0.5, hi[1] + 0.5
    t = np.where(rng.random(n) < 0.2, 2, 1).astype(np.int32)
    coeffs = {(1, 1): (1.0, 1.0, 2.5), (1, 2): (1.5, 0.8, 2.0), (2, 2): (0.5, 0.88, 2.2)}
    ref = M.Ref(M.LJ)
    ref.box(lo, hi, (1, 0, 1), ntypes=2)
    ref.add_atoms(x, t)
    ref.mass(1, 1.0)
    ref.mass(2, 1.0)
    ref.pair_lj(2.5)
    for (i, j), (e, s, c) in coeffs.items():
        ref.pair_coeff(i, j, e, s, c)
    ref.neighbor(0.3)
    ref.setup()
    ctx = mdx.Context(0)
    ctx.set_box(lo, hi, (1, 0, 1))
    ctx.set_atoms(x, t, np.array([0.0, 1.0, 1.0]), tags=np.arange(1, n + 1))
    ctx.pair_lj_from_coeffs(2, coeffs)
    ctx.position_format(fmt)
    ctx.neigh_modify(0.3)
    ctx.neigh_build()
    got, want = (np.sort(np.asarray(p, dtype=np.int64), axis=1) for p in (ctx.neigh_pairs(), ref.list_pairs()))
    assert ctx.stats()["total_neighbors"] == 2 * len(want)
    assert np.array_equal(np.sort(got[:, 0] << 32 | got[:, 1]), np.sort(want[:, 0] << 32 | want[:, 1]))
    ctx.close()


def test_collapsed_bin_is_reported_as_overflow():
    """2500 atoms in one bin with one = 2000: every one of them has more than
    `one` neighbours, the reference's "Neighbor list overflow"
    (neigh_half_bin.cpp:414-415); the build reports it as a status code
    after a bounded sort pass."""
    from lammps_amd import mdx
    x = _crowded(2500, 4)
    ctx = lj_context((0, 0, 0), (20.0, 20.0, 20.0), (1, 1, 1), x, mdx.FP64, one=2000)
    with pytest.raises(mdx.MdxError) as e:
        ctx.neigh_build()
    assert e.value.code == mdx.ERR_OVERFLOW and "boost neigh_modify one" in str(e.value)
    ctx.close()


def test_lost_atom_in_a_closed_box_is_reported():
    """boundary f: an atom outside the box is lost (the reference's
    'Lost atoms' check, thermo.cpp lost/error), an error and no crash"""
    from lammps_amd import mdx
    x = random_gas(20, 6.0, 0.9, seed=3) + 2.0
    ctx = lj_context((0, 0, 0), (10, 10, 10), (0, 0, 0), x, mdx.FP64)
    ctx.compute(1, 1)
    x2 = x.copy()
    x2[7, 1] = 10.5
    ctx.set_positions(x2)
    with pytest.raises(mdx.MdxError) as e:
        ctx.neigh_build()
    assert e.value.code == mdx.ERR_ARG and "Lost atoms" in str(e.value)
    ctx.close()


def _collapsing_droplet():
    """864 atoms of an fcc droplet expanded by 12% with inward velocities
    0.3 (x - centre), in a 30 sigma periodic box: the largest neighbour count
    goes from 54 to about 120 within 150 steps (the oracle on the same
    start), so a build inside the run needs more list capacity than the
    setup build sized."""
    a = (4.0 / 0.8442) ** (1.0 / 3.0) * 1.12
    basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    g = np.stack(np.meshgrid(*(np.arange(6),) * 3, indexing="ij"), -1).reshape(-1, 3)
    x = ((g[:, None] + basis[None]) * a).reshape(-1, 3)
    x = x - x.mean(0) + 15.0
    return x, -0.3 * (x - 15.0)


def test_list_regrows_inside_a_fused_run():
    """mdx_run's rebuilds queue the step behind the build before the host
    reads the build's flags; when the list outgrew its capacity that step
    does nothing and is queued again after the list is grown and rebuilt.
    The fused run (this path) and the unfused run (builds checked before
    the step) end bit for bit equal, with the same builds, and the capacity
    grew during the run."""
    from lammps_amd import mdx
    x, v = _collapsing_droplet()
    out = {}
    for fused in (True, False):
        ctx = mdx.Context(0)
        ctx.set_box((0, 0, 0), (30, 30, 30), (1, 1, 1))
        ctx.set_atoms(x, np.ones(len(x), dtype=np.int32), MASS, v=v, tags=np.arange(1, len(x) + 1))
        ctx.pair_lj_from_coeffs(1, {(1, 1): (1.0, 1.0, 2.5)})
        ctx.precision(mdx.FP64)
        ctx.neigh_modify(0.3, every=1, delay=0, check=True)
        ctx.fused(fused)
        ctx.setup()
        cap0 = ctx.stats()["capacity"]
        rows = ctx.run(200, 0.005, 1.0, 100)
        st = ctx.stats()
        out[fused] = dict(atoms=ctx.get_atoms(), rows=rows, st=st, cap0=cap0)
        ctx.close()
    for a, b in zip(out[True]["atoms"], out[False]["atoms"]):
        assert np.array_equal(a, b)
    st = out[True]["st"]
    assert st["ncalls"] == out[False]["st"]["ncalls"] > 10
    assert st["max_neighbors"] <= st["capacity"]
    assert st["capacity"] > out[True]["cap0"]
    assert len(out[True]["rows"]) == len(out[False]["rows"]) == 2
    for (s1, r1), (s2, r2) in zip(out[True]["rows"], out[False]["rows"]):
        assert s1 == s2
        np.testing.assert_allclose(r1, r2, rtol=1e-13, atol=1e-13 * max(abs(q) for q in r2))


def test_lost_atom_inside_a_fused_run_is_reported():
    """boundary f, an atom flying out mid-run: the step queued behind the
    build that finds it outside does nothing, and mdx_run returns the
    reference's 'Lost atoms' error"""
    from lammps_amd import mdx
    x = random_gas(20, 6.0, 0.9, seed=3) + 2.0
    v = np.zeros_like(x)
    v[np.argmax(x[:, 1]), 1] = 20.0  # the topmost atom, 0.1 sigma per step towards y = 10
    ctx = mdx.Context(0)
    ctx.set_box((0, 0, 0), (10, 10, 10), (0, 0, 0))
    ctx.set_atoms(x, np.ones(len(x), dtype=np.int32), MASS, v=v, tags=np.arange(1, len(x) + 1))
    ctx.pair_lj_from_coeffs(1, {(1, 1): (1.0, 1.0, 2.5)})
    ctx.precision(mdx.FP64)
    ctx.neigh_modify(0.3, every=1, delay=0, check=True)
    ctx.fused(True)
    ctx.setup()
    with pytest.raises(mdx.MdxError) as e:
        ctx.run(200, 0.005, 1.0, 0)
    assert e.value.code == mdx.ERR_ARG and "Lost atoms" in str(e.value)
    ctx.close()


def test_periodic_box_below_twice_the_cutoff_is_rejected():
    from lammps_amd import mdx
    x = random_gas(5, 5.0, 1.0, seed=4)
    ctx = lj_context((0, 0, 0), (5.0, 5.0, 5.0), (1, 1, 1), x, mdx.FP64)
    with pytest.raises(mdx.MdxError) as e:
        ctx.compute(1, 1)
    assert e.value.code == mdx.ERR_ARG and "2x the neighbour cutoff" in str(e.value)
    ctx.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("tpa", [4, 32])
def test_two_type_lj_matches_the_oracle(prec, tpa):
    """Kob-Andersen coefficients (two types, per-pair cutoffs): the general
    pair kernels (per-pair type lookups; single-type systems take a
    specialised path) against the oracle"""
    from lammps_amd import mdx
    L, n = 9.0, 600
    x = random_gas(n, L, 0.85, seed=11)
    t = np.where(np.random.default_rng(12).random(n) < 0.2, 2, 1).astype(np.int32)
    coeffs = {(1, 1): (1.0, 1.0, 2.5), (1, 2): (1.5, 0.8, 2.0), (2, 2): (0.5, 0.88, 2.2)}
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), (L, L, L), ntypes=2)
    ref.add_atoms(x, t)
    ref.mass(1, 1.0)
    ref.mass(2, 1.0)
    ref.pair_lj(2.5)
    for (i, j), (e, s, c) in coeffs.items():
        ref.pair_coeff(i, j, e, s, c)
    ref.neighbor(0.3)
    ref.setup()
    _, _, fref, _, _ = ref.state()
    eref, _ = ref.energy_virial()
    ctx = mdx.Context(0)
    ctx.set_box((0, 0, 0), (L, L, L), (1, 1, 1))
    ctx.set_atoms(x, t, np.array([0.0, 1.0, 1.0]), tags=np.arange(1, n + 1))
    ctx.pair_lj_from_coeffs(2, coeffs)
    ctx.precision(mdx.FP64 if prec == "fp64" else mdx.MIXED)
    ctx.neigh_modify(0.3)
    ctx.set_launch(0, tpa)
    out = ctx.compute(1, 1)
    mx, _ = force_errors(out["f"], fref)
    assert mx <= (1e-11 if prec == "fp64" else 1e-5)
    assert abs(out["eng"] - eref) <= (1e-11 if prec == "fp64" else 1e-6) * abs(eref)
    ctx.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_shifted_two_type_lj_energies_match_the_oracle(prec):
    """pair_modify shift yes (offset = the pair energy at the cutoff,
    pair_lj_cut.cpp:566-571) with per-pair cutoffs: total and per-atom
    energies, forces and virial against the oracle's"""
    from lammps_amd import mdx
    L, n = 9.0, 600
    x = random_gas(n, L, 0.85, seed=21)
    t = np.where(np.random.default_rng(22).random(n) < 0.3, 2, 1).astype(np.int32)
    coeffs = {(1, 1): (1.0, 1.0, 2.5), (1, 2): (1.5, 0.8, 2.0), (2, 2): (0.5, 0.88, 2.2)}
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), (L, L, L), ntypes=2)
    ref.add_atoms(x, t)
    ref.mass(1, 1.0)
    ref.mass(2, 1.0)
    ref.pair_lj(2.5, shift=True)
    for (i, j), (e, s, c) in coeffs.items():
        ref.pair_coeff(i, j, e, s, c)
    ref.neighbor(0.3)
    ref.setup()
    ref.compute(3, 5)
    fref = ref.state()[2]
    eref, wref = ref.energy_virial()
    ea_ref, va_ref = ref.peratom()
    ctx = mdx.Context(0)
    ctx.set_box((0, 0, 0), (L, L, L), (1, 1, 1))
    ctx.set_atoms(x, t, np.array([0.0, 1.0, 1.0]), tags=np.arange(1, n + 1))
    ctx.pair_lj_from_coeffs(2, coeffs, shift=True)
    ctx.precision(mdx.FP64 if prec == "fp64" else mdx.MIXED)
    ctx.neigh_modify(0.3)
    out = ctx.compute(3, 5, peratom=True)
    tol = 1e-11 if prec == "fp64" else 1e-5
    etol = 1e-11 if prec == "fp64" else 1e-6
    mx, _ = force_errors(out["f"], fref)
    assert mx <= tol
    assert abs(out["eng"] - eref) <= etol * abs(eref)
    np.testing.assert_allclose(out["virial"], wref, rtol=etol, atol=etol * np.abs(wref).max())
    np.testing.assert_allclose(out["eatom"], ea_ref, rtol=0, atol=100 * etol * np.abs(ea_ref).max())
    np.testing.assert_allclose(out["vatom"], va_ref, rtol=0, atol=100 * etol * np.abs(va_ref).max())
    ctx.close()


@pytest.mark.parametrize("style,n", [("lj", 3000), ("lj", 3001), ("lj", 10000), ("lj", 10001), ("lj", 40000),
                                     ("lj", 40001), ("lj", 48000), ("lj", 48001), ("eam", 6000), ("eam", 6001), ("eam", 10001), ("eam", 48001)])
def test_default_launch_shapes_agree_with_a_fixed_one(style, n):
    """On both sides of the sizes where the default launch shape changes:
    forces equal those of 8 lanes per atom in workgroups of 256 to the order
    of the sums (FP64: 1e-12 of the rms force)."""
    from gpu_helpers import CU_U3
    from lammps_amd import mdx
    rng = np.random.default_rng(n)
    cells = int(np.ceil((n / 4.0) ** (1.0 / 3.0)))
    a = (4.0 / 0.8442) ** (1.0 / 3.0) if style == "lj" else 3.615
    lo, hi, x = mdx.lattice("fcc", 0.8442 if style == "lj" else 3.615, "lj" if style == "lj" else "metal", (0, 0, 0),
                            (cells,) * 3)
    x = np.mod(x[rng.permutation(len(x))[:n]] + rng.uniform(-0.04 * a, 0.04 * a, (n, 3)), hi)
    ctx = mdx.Context(0)
    ctx.set_box(lo, hi, (1, 1, 1))
    ctx.set_atoms(x, np.ones(n, dtype=np.int32), np.array([0.0, 1.0 if style == "lj" else 63.55]))
    if style == "lj":
        ctx.pair_lj_from_coeffs(1, {(1, 1): (1.0, 1.0, 2.5)})
    else:
        mdx.eam_context_tables(ctx, CU_U3)
    ctx.neigh_modify(0.3 if style == "lj" else 1.0)
    ctx.precision(mdx.FP64)
    got = ctx.compute(1, 1)
    ctx.set_launch(256, 8)
    want = ctx.compute(1, 1)
    assert ctx.get_launch() == dict(block=256, tpa=8)
    assert force_errors(got["f"], want["f"])[0] <= 1e-12
    assert abs(got["eng"] - want["eng"]) <= 1e-12 * abs(want["eng"])
    ctx.close()


@pytest.mark.parametrize("n", [255, 1023, 1024, 1025])
def test_transfers_on_both_sides_of_the_mapped_memory_line(n):
    """Systems up to 1,024 atoms exchange positions and results through mapped
    host memory, larger ones through copies: what set_atoms took comes back
    unchanged, and forces, per-atom energies and virials match the oracle's."""
    from lammps_amd import mdx
    L = (n / 0.85) ** (1.0 / 3.0)
    x = random_gas(n, L, 0.8, seed=n)
    v = np.random.default_rng(n).normal(size=(n, 3))
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), (L, L, L))
    ref.add_atoms(x, np.ones(n, dtype=np.int32))
    ref.mass(1, 1.0)
    ref.pair_lj(2.5)
    ref.pair_coeff(1, 1, 1.0, 1.0, 2.5)
    ref.neighbor(0.3)
    ref.setup()
    ref.compute(3, 5)
    ea, va = ref.peratom()
    ctx = mdx.Context(0)
    ctx.set_box((0, 0, 0), (L, L, L), (1, 1, 1))
    ctx.set_atoms(x, np.ones(n, dtype=np.int32), MASS, v=v)
    ctx.pair_lj_from_coeffs(1, {(1, 1): (1.0, 1.0, 2.5)})
    ctx.neigh_modify(0.3)
    gx, gv, gf, gi = ctx.get_atoms()
    assert np.array_equal(gx, x) and np.array_equal(gv, v) and not gf.any() and not gi.any()
    for _ in range(2):  # the second call after a position update
        out = ctx.compute(3, 5, peratom=True)
        assert force_errors(out["f"], ref.state()[2])[0] <= 1e-11
        np.testing.assert_allclose(out["eatom"], ea, rtol=0, atol=1e-10 * np.abs(ea).max())
        np.testing.assert_allclose(out["vatom"], va, rtol=0, atol=1e-10 * np.abs(va).max())
        ctx.set_positions(x)
        ctx.set_positions(x)
    ctx.close()


def test_atoms_handed_over_again_give_what_a_fresh_context_gives():
    """set_atoms keeps storage that fits: growing, shrinking and regrown atom
    counts, changed density, types and velocities in one context, each against
    a context of its own."""
    from lammps_amd import mdx

    def forces(ctx, k, n, L, ntypes):
        rng = np.random.default_rng(k)
        x = random_gas(n, L, 0.8, seed=k)
        t = rng.integers(1, ntypes + 1, n).astype(np.int32)
        ctx.set_box((0, 0, 0), (L, L, L), (1, 1, 1))
        ctx.set_atoms(x, t, np.ones(ntypes + 1), v=None if k % 2 else x)
        ctx.pair_lj_from_coeffs(ntypes, {(i, i): (1.0, 1.0, 2.5) for i in range(1, ntypes + 1)})
        ctx.neigh_modify(0.3)
        ctx.precision(mdx.MIXED if k % 3 == 0 else mdx.FP64)
        out = ctx.compute(3, 5, peratom=True)
        return [out["f"], out["eatom"], out["vatom"], np.array([out["eng"]])] + list(ctx.get_atoms())

    kept = mdx.Context(0)
    for k, (n, L, nt) in enumerate([(3000, 16.0, 1), (2900, 15.5, 1), (3072, 40.0, 1), (1600, 13.0, 1), (1400, 12.5, 1),
                                    (2999, 15.5, 1), (700, 9.5, 1), (1200, 12.0, 1)]):
        fresh = mdx.Context(0)
        for a, b in zip(forces(kept, k, n, L, nt), forces(fresh, k, n, L, nt)):
            assert np.array_equal(a, b), (k, n)
        fresh.close()
    kept.close()


@pytest.mark.parametrize("bad", [0, -3, 2, 1 << 20])
def test_noalloc_refuses_types_out_of_range(bad):
    """One type outside 1..ntypes in device memory: an error, the force array
    left as it was; the context computes on afterwards."""
    import torch
    from lammps_amd import mdx
    rng = np.random.default_rng(4)
    lo, hi, x = mdx.lattice("fcc", 0.8442, "lj", (0, 0, 0), (6, 6, 6))
    x = np.mod(x + rng.uniform(-0.05, 0.05, x.shape), hi)
    n = len(x)
    ctx = lj_context((0, 0, 0), hi, (1, 1, 1), x, mdx.FP64)
    xd = torch.tensor(x, device="cuda:0")
    t = np.ones(n, dtype=np.int32)
    t[n - 5] = bad
    td = torch.tensor(t, device="cuda:0")
    fd = torch.full((n, 3), 7.0, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    with pytest.raises(mdx.MdxError, match="type out of range") as e:
        ctx.compute_noalloc(n, xd.data_ptr(), td.data_ptr(), fd.data_ptr())
    assert e.value.code == mdx.ERR_ARG
    assert bool((fd == 7.0).all())
    td[n - 5] = 1
    torch.cuda.synchronize()
    eng, _ = ctx.compute_noalloc(n, xd.data_ptr(), td.data_ptr(), fd.data_ptr())
    out = ctx.compute(1, 1)
    assert force_errors(fd.cpu().numpy() - 7.0, out["f"])[0] <= 1e-12
    assert abs(eng - out["eng"]) <= 1e-12 * abs(out["eng"])
    ctx.close()


def copper(cells, seed, amp=0.1):
    """fcc copper with atoms displaced by up to amp: box and wrapped positions."""
    from lammps_amd import mdx
    lo, hi, x = mdx.lattice("fcc", 3.615, "metal", (0, 0, 0), cells)
    x = x + np.random.default_rng(seed).uniform(-amp, amp, x.shape)
    return np.asarray(lo), np.asarray(hi), np.mod(x, hi)


def eam_pair(path, hi, x, skin=1.0):
    """One system of one-element eam atoms in the oracle (set up) and in a context (FP64)."""
    from lammps_amd import mdx
    ref = M.Ref(M.METAL)
    ref.box((0, 0, 0), hi)
    ref.add_atoms(x, np.ones(len(x), dtype=np.int32))
    ref.pair_eam(path)
    ref.neighbor(skin)
    ref.setup()
    ref.compute(3, 5)
    ctx = mdx.Context(0)
    ctx.set_box((0, 0, 0), hi, (1, 1, 1))
    ctx.set_atoms(x, np.ones(len(x), dtype=np.int32), np.array([0.0, 63.55]))
    mdx.eam_context_tables(ctx, path)
    ctx.neigh_modify(skin)
    return ref, ctx


@pytest.mark.parametrize("tpa", [4, 8, 16, 32])
def test_coincident_eam_atoms_have_the_density_of_zero_separation(tpa):
    """Two atoms in one place (FP64, spline tables in LDS and not): densities,
    and the forces and energies of all other atoms, are the oracle's; the
    pair's energy is infinite there and here."""
    from gpu_helpers import CU_U3
    lo, hi, x = copper((5, 5, 4), 11)
    x[137] = x[21]
    ref, ctx = eam_pair(CU_U3, hi, x)
    ctx.set_launch(256, tpa)
    out = ctx.compute(3, 5, peratom=True)
    rho, fp = ctx.eam_rho_fp()
    rho_ref, fp_ref = ref.eam_rho_fp()
    assert np.isfinite(rho_ref).all()
    np.testing.assert_allclose(rho, rho_ref, rtol=1e-11)
    np.testing.assert_allclose(fp, fp_ref, rtol=0, atol=1e-10 * np.abs(fp_ref).max())
    rest = np.setdiff1d(np.arange(len(x)), [21, 137])
    assert force_errors(out["f"][rest], ref.state()[2][rest])[0] <= 1e-11
    ea = ref.peratom()[0]
    np.testing.assert_allclose(out["eatom"][rest], ea[rest], rtol=0, atol=1e-10 * np.abs(ea[rest]).max())
    assert ref.energy_virial()[0] == np.inf and out["eng"] == np.inf
    ctx.close()


@pytest.mark.parametrize("style,cells", [("lj", 5), ("lj", 15), ("lj", 23), ("eam", 6), ("eam", 14), ("eam", 22)])
@pytest.mark.parametrize("prec", [0, 1])
def test_default_launch_shape_can_be_set_by_value(style, cells, prec):
    """What get_launch reports can be handed to set_launch and is then in
    force, and gives the same forces; other blocks above 256 stay refused."""
    from gpu_helpers import CU_U3
    from lammps_amd import mdx
    if style == "lj":
        lo, hi, x = mdx.lattice("fcc", 0.8442, "lj", (0, 0, 0), (cells,) * 3)
        ctx = lj_context((0, 0, 0), hi, (1, 1, 1), np.mod(x + 0.01, hi), prec)
    else:
        lo, hi, x = copper((cells,) * 3, 2)
        ctx = mdx.Context(0)
        ctx.set_box((0, 0, 0), hi, (1, 1, 1))
        ctx.set_atoms(x, np.ones(len(x), dtype=np.int32), np.array([0.0, 63.55]))
        mdx.eam_context_tables(ctx, CU_U3)
        ctx.precision(prec)
        ctx.neigh_modify(1.0)
    f = ctx.compute(0, 0)["f"]
    shape = ctx.get_launch()
    ctx.set_launch(**shape)
    assert ctx.get_launch() == shape
    assert np.array_equal(ctx.compute(0, 0)["f"], f)
    for block in (320, 384, 448, 576, 1024, 96):
        with pytest.raises(mdx.MdxError):
            ctx.set_launch(block, 8)
    assert ctx.get_launch() == shape
    # 512 threads are the FP64 eam kernels' with tables in LDS; others run 256
    ctx.set_launch(512, 8)
    assert ctx.get_launch() == dict(block=512 if style == "eam" and prec == mdx.FP64 else 256, tpa=8)
    ctx.set_launch(256, 8)
    want = ctx.compute(0, 0)["f"]
    ctx.set_launch(512, 8)
    assert np.array_equal(ctx.compute(0, 0)["f"], want)
    tuned = ctx.autotune(2)
    ctx.set_launch(**tuned)
    assert ctx.get_launch() == tuned
    ctx.close()


@pytest.mark.parametrize("prec,nr", [("fp64", 799), ("fp64", 800), ("mixed", 1023), ("mixed", 1024)])
@pytest.mark.parametrize("tpa", [4, 8, 16])
def test_eam_tables_on_both_sides_of_the_lds_limits(prec, nr, tpa, tmp_path):
    """One-element tables of the largest size that goes to LDS (800 knots in
    FP64, 1,024 mixed, the unused knot 0 included) and one knot more: forces,
    per-atom energies and virials are the oracle's."""
    from lammps_amd import mdx
    path = str(tmp_path / "cu.eam")
    mdx.write_synthetic_funcfl(path, nr=nr, dr=4.99 / (nr - 1))
    lo, hi, x = copper((6, 5, 5), nr)
    ref, ctx = eam_pair(path, hi, x)
    ctx.precision(mdx.FP64 if prec == "fp64" else mdx.MIXED)
    ea, va = ref.peratom()
    ftol, etol = (1e-11, 1e-10) if prec == "fp64" else (1e-5, 1e-5)
    for block in (256, 512):
        ctx.set_launch(block, tpa)
        out = ctx.compute(3, 5, peratom=True)
        assert force_errors(out["f"], ref.state()[2])[0] <= ftol
        np.testing.assert_allclose(out["eatom"], ea, rtol=0, atol=etol * np.abs(ea).max())
        np.testing.assert_allclose(out["vatom"], va, rtol=0, atol=etol * np.abs(va).max())
    ctx.close()


@pytest.mark.parametrize("n", [1024, 1025, 97000])
def test_moved_positions_are_computed_on_the_old_list(n):
    """Positions handed over again after a move below half the skin, through
    mapped memory, one staged piece and several: forces, per-atom energies and
    virials are the oracle's at the new positions."""
    from lammps_amd import mdx
    rng = np.random.default_rng(n)
    cells = int(np.ceil((n / 4.0) ** (1.0 / 3.0)))
    lo, hi, x = mdx.lattice("fcc", 0.8442, "lj", (0, 0, 0), (cells,) * 3)
    x = np.mod(x[rng.permutation(len(x))[:n]] + rng.uniform(-0.05, 0.05, (n, 3)), hi)
    ctx = lj_context((0, 0, 0), hi, (1, 1, 1), x, mdx.FP64)
    first = ctx.compute(3, 5, peratom=True)
    builds = ctx.stats()["total_neighbors"]
    moved = x + rng.uniform(-0.08, 0.08, x.shape)
    ctx.set_positions(moved)
    out = ctx.compute(3, 5, peratom=True)
    assert ctx.stats()["total_neighbors"] == builds
    ref = M.Ref(M.LJ)
    ref.box((0, 0, 0), hi)
    ref.add_atoms(np.mod(moved, hi), np.ones(n, dtype=np.int32))
    ref.mass(1, 1.0)
    ref.pair_lj(2.5)
    ref.pair_coeff(1, 1, 1.0, 1.0, 2.5)
    ref.neighbor(0.3)
    ref.setup()
    ref.compute(3, 5)
    ea, va = ref.peratom()
    f = ref.state()[2]
    assert force_errors(first["f"], f)[0] > 1e-3  # the move changes the forces
    assert force_errors(out["f"], f)[0] <= 1e-11
    np.testing.assert_allclose(out["eatom"], ea, rtol=0, atol=1e-10 * np.abs(ea).max())
    np.testing.assert_allclose(out["vatom"], va, rtol=0, atol=1e-10 * np.abs(va).max())
    ctx.close()


@pytest.mark.parametrize("style,ntypes", [("lj", 1), ("lj", 2), ("eam", 1)])
@pytest.mark.parametrize("fmt", [0, 1])
def test_mixed_forces_have_the_same_bits_at_four_and_eight_lanes(style, ntypes, fmt):
    """The default takes four lanes per atom above 40,000 atoms and eight
    below: a mixed trajectory must not depend on which."""
    from gpu_helpers import CU_U3
    from lammps_amd import mdx
    rng = np.random.default_rng(ntypes)
    ctx = mdx.Context(0)
    if style == "lj":
        lo, hi, x = mdx.lattice("fcc", 0.8442, "lj", (0, 0, 0), (11, 12, 10))
        x = np.mod(x + rng.uniform(-0.1, 0.1, x.shape), hi)[:-3]
        ctx.set_box((0, 0, 0), hi, (1, 1, 1))
        ctx.set_atoms(x, rng.integers(1, ntypes + 1, len(x)).astype(np.int32), np.ones(ntypes + 1))
        ctx.pair_lj_from_coeffs(ntypes, {(1, 1): (1.0, 1.0, 2.5), (ntypes, ntypes): (0.5, 0.88, 2.2)})
        ctx.neigh_modify(0.3)
    else:
        lo, hi, x = copper((9, 10, 8), 5)
        ctx.set_box((0, 0, 0), hi, (1, 1, 1))
        ctx.set_atoms(x[:-3], np.ones(len(x) - 3, dtype=np.int32), np.array([0.0, 63.55]))
        mdx.eam_context_tables(ctx, CU_U3)
        ctx.neigh_modify(1.0)
    ctx.position_format(fmt)
    ctx.precision(mdx.MIXED)
    got = []
    for tpa in (4, 8):
        ctx.set_launch(256, tpa)
        got.append([ctx.compute(0, 0)["f"]] + (list(ctx.eam_rho_fp()) if style == "eam" else []))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    ctx.close()
