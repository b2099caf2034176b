"""A device allocation that fails is an error and nothing worse: the call
returns it, and whatever the program calls next either works or returns an
error too - no kernel is launched on an array that is not there.

CPU only.  The library runs in a child process on tests/sanitize/fake_hip.cpp
(a HIP runtime whose kernels do nothing and that checks the pointers they are
given).  A sequence of calls is run once for each of its allocations, with
that one failing; after the error the calls so far, smaller ones among them,
are made again and have to succeed."""
import ctypes
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))
HIP_INCLUDE = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(HIP_INCLUDE, "hip")),
                                reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I" + HIP_INCLUDE,
                        os.path.join(HERE, "sanitize", "fake_hip.cpp"), "-o", lib], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return lib


@pytest.mark.parametrize("what", ["batch_lj", "batch_eam", "context_lj", "context_eam", "context_run"])
def test_each_allocation_failing_once(fake, what):
    preload = " ".join(q for q in (fake, os.environ.get("LD_PRELOAD")) if q)
    env = dict(os.environ, LD_PRELOAD=preload, FAKE_HIP=fake, MDX_HIP_RUNTIME="rocm", PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), what], capture_output=True, text=True, env=env,
                       timeout=300)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "allocations failed in turn" in r.stdout


# ------------------------------------------------------------ the child process

def _sequences():
    import numpy as np

    from lammps_amd import batch as B
    from lammps_amd import mdx
    from lammps_amd import workloads as W
    fk = ctypes.CDLL(os.environ["FAKE_HIP"])
    rng = np.random.default_rng(1)
    one = np.ones((3, 3))
    x = rng.uniform(0.0, 20.0, (500, 3))
    G = rng.normal(size=x.shape)

    def batch():
        fk.fake_rows(40)
        b = B.Batch([300, 200], [[0, 0, 0]] * 2, [[20, 20, 20]] * 2, [[1, 1, 1]] * 2, 2, np.ones(500, np.int32))
        b.set_positions(x)
        return b

    def knots(b, n):
        p = W.synthetic_knots(n)
        b.eam_init(p["drho"], p["dr"], p["cut"], p["frho"], p["rhor"], p["z2r"])

    def many_rows(b, n, skin):  # a longer largest row, seen by a new list
        fk.fake_rows(n)
        b.skin(skin)
        b.neigh_stats()

    def context(n=400):
        fk.fake_rows(10)
        c = mdx.Context(0)
        c.set_box((0, 0, 0), (30, 30, 30), (1, 1, 1))
        c.neigh_modify(0.3, every=1, delay=0, check=False)
        atoms(c, n)
        return c

    def atoms(c, n):
        c.set_atoms(np.random.default_rng(n).uniform(0.0, 30.0, (n, 3)), np.ones(n, np.int32), np.array([0.0, 1.0]))

    def lj(c):
        c.pair_lj_from_coeffs(1, {(1, 1): (1.0, 1.0, 2.5)})

    def eam(c, scale=1):
        t = mdx.eam_funcfl(os.path.join(ROOT, "tests", "golden", "Cu_u3.eam"))
        z = np.zeros(4, dtype=np.int32)
        c.pair_eam(1, t["nrho"], t["drho"], t["nr"], t["dr"], t["rhomax"], 4.95 ** 2,
                   np.repeat(t["frho_spline"], scale, axis=0), t["rhor_spline"], t["z2r_spline"], z[:2], z, z)

    def grown(c, n):  # a list with more entries per atom, in the middle of a run
        fk.fake_rows(n)
        c.run(3, 0.001)

    def wide(c, L):  # more bins
        c.set_box((0, 0, 0), (L, L, L), (1, 1, 1))
        c.compute(1, 1)

    small, large = one * 2.0, one * 2.5
    return fk, {
        "batch_lj": (batch, [
            lambda b: b.lj_init(one, one, large), lambda b: b.lj_forces(), lambda b: b.lj_vjp(G),
            lambda b: many_rows(b, 150, 0.1), lambda b: b.lj_forces(), lambda b: many_rows(b, 100, 0.2),
            lambda b: (b.lj_init(one, one, small), b.lj_forces(), b.lj_vjp(G)),  # more bins
        ]),
        "batch_eam": (batch, [
            lambda b: knots(b, 32), lambda b: b.eam_forces(), lambda b: b.eam_vjp(G),
            lambda b: knots(b, 64), lambda b: b.eam_forces(), lambda b: b.eam_vjp(G),
            lambda b: (b.lj_init(one, one, large), b.lj_vjp(G)), lambda b: knots(b, 64), lambda b: b.eam_vjp(G),
        ]),
        "context_lj": (context, [
            lj, lambda c: c.compute(1, 1), lambda c: c.compute(3, 5, peratom=True), lambda c: wide(c, 80.0),
            lambda c: wide(c, 170.0),  # beyond the one-workgroup scan
            lambda c: atoms(c, 900), lambda c: c.compute(1, 1), lambda c: atoms(c, 420), lambda c: c.compute(1, 1),
            lambda c: c.get_atoms(),
        ]),
        "context_eam": (context, [
            eam, lambda c: c.compute(1, 1), lambda c: eam(c, 3), lambda c: c.compute(3, 5, peratom=True),
            lambda c: c.eam_rho_fp(),
        ]),
        "context_run": (context, [
            lj, lambda c: c.run(3, 0.001), lambda c: grown(c, 300), lambda c: c.run(2, 0.001),
            lambda c: grown(c, 700), lambda c: c.run(2, 0.001),
        ]),
    }


def _child(what):
    from lammps_amd import mdx
    fk, seqs = _sequences()
    make, ops = seqs[what]
    n = 0
    while True:
        n += 1
        fk.fake_fail_in(n)
        failed = None
        try:
            obj = make()
        except mdx.MdxError as e:  # nothing came to be
            assert e.code == mdx.ERR_NOMEM, e
            continue
        for k, op in enumerate(ops):
            try:
                op(obj)
            except mdx.MdxError as e:
                assert failed is None and e.code == mdx.ERR_NOMEM, (n, k, str(e))
                failed = k
                try:
                    op(obj)  # the call that failed, again
                except mdx.MdxError as again:
                    # an init that failed leaves no pair style; anything else works now
                    assert again.code == mdx.ERR_ARG, (n, k, str(again))
                for q in ops[:k + 1]:
                    q(obj)
        obj.close()
        assert fk.fake_bad() == 0, (what, "allocation", n, "operation", failed)
        if failed is None:
            break
    assert n > 10
    print("%s: %d allocations failed in turn, %d launches" % (what, n - 1, fk.fake_launches()))


if __name__ == "__main__":
    _child(sys.argv[1])
