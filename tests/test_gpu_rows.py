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
    s = OMMPSystem.from_arrays(spec["amoeba"], spec["cmm"], spec["q"], spec["pol"], spec["bonds_ri"],
                               spec["bonds_ci"], pgroup=spec["pgroup"] if spec["amoeba"] else None)
    q = spec["q"].copy()
    if spec["amoeba"]:
        q[:, 4:10] /= 3.0
        scales = [[0, 0, .4, .8], [0, 0, 1, 1], [0, 1, 1, 1], [1, 1, 1, 1], [0, 0, .5, 1]]
    else:
        scales = [[0, 0, 1, 1]] * 4 + [[1, 1, 1, 1]]
    n = len(spec["pol"])
    o = oa.OracleSystem(dict(nmm=n, amoeba=spec["amoeba"], cmm=spec["cmm"], q=q, pol=spec["pol"],
                             adj_ri=spec["bonds_ri"], adj_ci=spec["bonds_ci"], grp=spec["pgroup"],
                             td=np.full(n, 0.39), scales=np.array(scales, dtype=float),
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
