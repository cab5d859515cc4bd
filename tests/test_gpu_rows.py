"""The per-target T matvec (one workgroup per 1 to 8 targets, the threads on the
sources) against the oracle at the edges of its tiles: one and two sites, around
one wave, one workgroup of sources and the sizes where the number of targets
changes, with remainders of targets; both precisions, one and two columns, AMOEBA
and AMBER (Wang, with screened pairs).  Bars: FP64 a sum of up to 3,003 pairs
rounds to ~sqrt(3003) eps = 1.2e-14 of the largest component, 1e-13 asked; FP32
~3003^0.5 * 6e-8 = 3.3e-6 of a typical term at most, 2e-6 of the largest component asked
(as the other FP32 sweeps)."""
import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


def chain(n, amoeba, seed=5):
    """n sites on a jittered lattice, bonded in runs of 7."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.arange(side)
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1).reshape(-1, 3)[:n] * 4.0
    p = p + rng.uniform(-0.8, 0.8, size=p.shape)
    bonded = (np.arange(n - 1) % 7) != 6
    nb = [[k for k, ok in ((i - 1, i > 0 and bonded[i - 1]), (i + 1, i < n - 1 and bonded[min(i, n - 2)])) if ok]
          for i in range(n)]
    ri = np.concatenate([[0], np.cumsum([len(r) for r in nb])]).astype(np.int32)
    ci = np.array([v for r in nb for v in r], dtype=np.int32)
    q = rng.normal(0.0, 0.2, size=(n, 10))
    q[:, 6] -= q[:, 4] + q[:, 6] + q[:, 9]
    return dict(amoeba=amoeba, cmm=p, q=q if amoeba else q[:, :1], pol=rng.uniform(2.0, 9.0, size=n), bonds_ri=ri,
                bonds_ci=ci, pgroup=(np.arange(n) // 7).astype(np.int32))


def pair(spec):
    from openmmpol_amd import OMMPSystem
    td = spec.get("td", np.full(len(spec["pol"]), 0.39))
    s = OMMPSystem.from_arrays(spec["amoeba"], spec["cmm"], spec["q"], spec["pol"], spec["bonds_ri"],
                               spec["bonds_ci"], pgroup=spec["pgroup"] if spec["amoeba"] else None,
                               thole_a=spec.get("td"))
    q = spec["q"].copy()
    if spec["amoeba"]:
        q[:, 4:10] /= 3.0
        scales = [[0, 0, .4, .8], [0, 0, 1, 1], [0, 1, 1, 1], [1, 1, 1, 1], [0, 0, .5, 1]]
    else:
        scales = [[0, 0, 1, 1]] * 4 + [[1, 1, 1, 1]]
    n = len(spec["pol"])
    o = oa.OracleSystem(dict(nmm=n, amoeba=spec["amoeba"], cmm=spec["cmm"], q=q, pol=spec["pol"],
                             adj_ri=spec["bonds_ri"], adj_ci=spec["bonds_ci"], grp=spec["pgroup"],
                             td=td, scales=np.array(scales, dtype=float),
                             thole_scale=0.0 if spec["amoeba"] else 2.5874))
    return s, o


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 255, 257, 512, 513, 3000, 3001, 3003])
def test_per_target_matvec(n, amoeba):
    s, o = pair(chain(n, amoeba))
    x = np.random.default_rng(n).normal(0.0, 0.05, size=(2, n, 3))
    want = np.stack([o.tmatvec(x[0]), o.tmatvec(x[1])])
    for kind, tol in (("plain64", 1e-13), ("plain32", 2e-6)):
        for ncols in (1, 2):
            y, _ = s.tmatvec(x[:ncols], kind=kind)
            assert np.abs(y - want[:ncols]).max() <= tol * np.abs(want).max(), (kind, ncols)
        assert np.array_equal(s.tmatvec(x, kind=kind)[0], y)
    s.terminate()


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("n,kinds", [(n, ("sym64", "sym32")) for n in (1, 33, 64, 65, 129, 255, 257, 449, 513, 769)]
                         + [(3001, ("plain64", "plain32", "sym64", "sym32"))])
@pytest.mark.parametrize("scale", [1.0, 0.35])
def test_damping_cutoff(n, kinds, scale, amoeba):
    """The pair-once sweep (diagonal and other block pairs, partly filled sub-tiles)
    and the per-target one with its lists of damped pairs, at 4 bohr and at 1.4 bohr
    spacing (hundreds of damped pairs a site: the lists overflow), with one outlying
    polarizability, against the oracle.  FP64: 3,001 terms of rounding 1.1e-16 on
    sums that cancel to a few of them: 1e-12 of the largest component; FP32 by its
    rounding of 6e-8: 3e-4 at 1.4 bohr, and 2e-6 at 4 bohr, where they do not cancel."""
    spec = chain(n, amoeba)
    spec["cmm"] = spec["cmm"] * scale
    spec["pol"][n // 2] = 300.0
    s, o = pair(spec)
    x = np.random.default_rng(n).normal(0.0, 0.05, size=(2, n, 3))
    want = np.stack([o.tmatvec(x[0]), o.tmatvec(x[1])])
    for kind in kinds:
        for ncols in (1, 2):
            y, _ = s.tmatvec(x[:ncols], kind=kind)
            bar = 1e-12 if kind.endswith("64") else 2e-6 if scale == 1.0 else 3e-4
            assert np.abs(y - want[:ncols]).max() <= bar * np.abs(want).max(), (kind, ncols)
        assert np.array_equal(s.tmatvec(x, kind=kind)[0], y)
    s.terminate()


@pytest.mark.parametrize("a", [0.0, -0.4])
@pytest.mark.parametrize("n", [300, 3001])
def test_damping_factor_not_positive(n, a):
    """AMOEBA damping factors that bound no distance: 0 damps every pair of its site
    to nothing, a negative one lets its pairs grow with the distance (per-target sweep
    alone: they overflow beyond some 20 bohr).  FP64 against the oracle, 1e-12 of the largest component (3,001 terms of rounding 1.1e-16,
    and of an exponential's argument of up to ~280: 280 eps = 6e-14)."""
    spec = chain(n, True)
    spec["td"] = np.full(n, 0.39)
    spec["td"][n // 2] = a
    if a < 0.0:
        spec["cmm"] = spec["cmm"] * (0.35 if n == 300 else 0.2)
    s, o = pair(spec)
    x = np.random.default_rng(n).normal(0.0, 0.05, size=(2, n, 3))
    want = np.stack([o.tmatvec(x[0]), o.tmatvec(x[1])])
    assert np.isfinite(want).all()
    for kind in ("plain64", "sym64")[:1 if a < 0.0 else 2]:
        y, _ = s.tmatvec(x, kind=kind)
        assert np.abs(y - want).max() <= 1e-12 * np.abs(want).max(), kind
    s.terminate()


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("n", [1, 15, 17, 260, 1030])
def test_thin_source_splits(n, amoeba):
    """The static field and the gradient with sources split down to 16 per
    workgroup (one site, one split short or past full, several target blocks)
    against the oracle; bars as the larger systems' (1e-12 and 1e-11 of the
    largest component: sums of at most 1,030 pairs)."""
    s, o = pair(chain(n, amoeba))
    e, eo = s.e_m2d, o.m2d()
    assert np.abs(e - eo).max() <= 1e-12 * max(np.abs(eo).max(), 1e-300)
    s.set_external_field(np.random.default_rng(n).normal(0.0, 1e-2, size=(n, 3)))
    g = s.polelec_geomgrad()
    want = o.polelec_geomgrad(np.array(s.ipd))
    assert np.abs(g - want).max() <= 1e-11 * max(np.abs(want).max(), 1e-300)
    s.terminate()


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("npoints", [1, 2047, 2049, 8193, 16383, 16385])
def test_external_points(npoints, amoeba):
    """Potential and field at external points around the sizes where the points
    per thread and the source splits change, against the oracle (1e-12 of the
    largest value: 300 sources)."""
    n = 300
    s, o = pair(chain(n, amoeba))
    s.set_external_field(np.zeros((n, 3)))
    ipd = np.array(s.ipd)
    rng = np.random.default_rng(npoints)
    c = rng.uniform(-30.0, -2.5, size=(npoints, 3))
    for name, which in (("mm", 1), ("pol", 2), ("mmpol", 3)):
        v, e = o.x2e(c, which, ipd)
        got = getattr(s, f"potential_{name}2ext")(c)
        assert np.abs(got - v).max() <= 1e-12 * np.abs(v).max(), name
        got = getattr(s, f"field_{name}2ext")(c)
        assert np.abs(got - e).max() <= 1e-12 * np.abs(e).max(), name
    s.terminate()


@pytest.mark.parametrize("n,spacing", [(1, 4.0), (2, 4.0), (161, 4.0), (700, 3.0), (125, 0.9)])
def test_neighbour_lists(n, spacing):
    """The near-field preconditioner (lists built with the device's grid) against
    2 alpha r - alpha T_near alpha r from the oracle's dense T, before and after a
    change of coordinates: no neighbours, a few, rows longer than the 64 gathered
    at once.  FP32 tensors: 2e-6 of the largest component, as the 3,000-site test."""
    spec = chain(n, True, seed=8)
    rng = np.random.default_rng(9)
    cut = 3.0 * 1.8897261245650
    s = None
    for scale in (1.0, 1.13):
        spec["cmm"] = spec["cmm"] / (4.0 if scale == 1.0 else spacing) * spacing * scale
        if s is None:
            s, o = pair(spec)
        else:
            s.update_coordinates(spec["cmm"])
            o = pair(spec)[1]
        d = np.linalg.norm(spec["cmm"][:, None] - spec["cmm"][None], axis=2)
        near = (d < cut) & (d > 0.0)
        if n == 125:
            assert near.sum(axis=1).max() > 64
        al = np.repeat(spec["pol"], 3)
        T = np.where(np.repeat(np.repeat(near, 3, 0), 3, 1), o.tmat(), 0.0)
        r = rng.normal(size=(2, n, 3))
        want = np.array([2.0 * al * v - al * (T @ (al * v)) for v in r.reshape(2, -1)]).reshape(2, n, 3)
        z, on = s.inner_precond_apply(r)
        assert on and np.abs(z - want).max() <= 2e-6 * np.abs(want).max()
    s.terminate()


@pytest.mark.parametrize("n", [10, 300])
def test_coincident_sites_are_refused(n):
    """Two atoms at one point end the process with the reference's message, on the
    host's check (10 atoms) and on the grid's (300)."""
    import os
    import subprocess
    import sys
    code = ("import sys; sys.path[:0] = ['tests', '.']; import numpy as np, test_gpu_rows as t\n"
            f"spec = t.chain({n}, True); spec['cmm'][{n - 3}] = spec['cmm'][1]\n"
            "s, _ = t.pair(spec); print('built', flush=True)\n"
            f"s.set_external_field(np.zeros(({n}, 3))); print('solved')\n")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=100)
    assert p.returncode == 1 and "built" in p.stdout and "solved" not in p.stdout
    assert "two atoms placed in the same point" in p.stdout + p.stderr
