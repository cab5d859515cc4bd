"""The matrix-core transfer and T matvec of the fast multipoles (orders up to 8)
on small trees: one leaf, two per side (no far field), and far fields of two and
three levels, leaves of 6 to 141 sites (from 97 on 32 targets share a
workgroup), odd sizes, orders whose coefficients fill 1 to 5 tiles; AMOEBA and
AMBER.  Against the complex kernels, which an order of the static field above 8
selects and which sum the same truncated expansions in another order: 1e-12 of
the largest component (FP64 sums of a few thousand terms); and with no far field
against the direct matvec, 1e-13."""
import numpy as np
import pytest

from test_gpu_rows import chain

pytestmark = pytest.mark.gpu


def _system(n, amoeba):
    from openmmpol_amd import OMMPSystem
    spec = chain(n, amoeba, seed=n)
    return OMMPSystem.from_arrays(amoeba, spec["cmm"], spec["q"], spec["pol"], spec["bonds_ri"], spec["bonds_ci"],
                                  pgroup=spec["pgroup"] if amoeba else None)


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("n,cell", [(7, 40.0), (301, 12.0), (1003, 8.0), (3001, 7.0), (9001, 20.0)])
def test_matvec_small_trees(n, cell, amoeba):
    s = _system(n, amoeba)
    x = np.random.default_rng(3).normal(0.0, 0.05, size=(2, n, 3))
    want, _ = s.tmatvec(x, kind="plain64")
    scale = np.abs(want).max()
    for p in (2, 4, 6, 8):
        s.enable_fmm(lmax=p, lmax_pol=p, distance=1.0, min_cell_size=cell)
        y, _ = s.tmatvec(x, kind="fmm")
        assert np.array_equal(s.tmatvec(x, kind="fmm")[0], y)
        one, _ = s.tmatvec(x[:1], kind="fmm")
        assert np.array_equal(one, y[:1])
        s.enable_fmm(lmax=9, lmax_pol=p, distance=1.0, min_cell_size=cell)
        old, _ = s.tmatvec(x, kind="fmm")
        assert np.abs(y - old).max() <= 1e-12 * scale, p
        if n == 7:
            assert np.abs(y - want).max() <= 1e-13 * scale
    s.terminate()


@pytest.mark.parametrize("p", [1, 3, 5, 7, 8])
def test_static_field_and_gradient_orders(p):
    """The static field and the gradient through the transfer against the complex
    kernels (selected by an order of 9 for the other of the two expansions where
    the pass allows it: the gradient runs at the larger of the two orders, so it
    is compared at 8 and 9 through the truncation error against the direct one)."""
    n = 3001
    s = _system(n, True)
    direct = s.e_m2d
    s.set_solver_tolerance(1e-10, 500)
    s.set_external_field(np.zeros((n, 3)))
    gd = s.polelec_geomgrad()
    s.enable_fmm(lmax=p, lmax_pol=p, distance=1.0, min_cell_size=7.0)
    new = s.e_m2d
    s.enable_fmm(lmax=p, lmax_pol=9, distance=1.0, min_cell_size=7.0)
    old = s.e_m2d
    scale = np.abs(direct).max()
    assert np.abs(new - old).max() <= 1e-12 * scale
    if p == 8:
        err = []
        for q in (4, 8, 9):
            s.enable_fmm(lmax=q, lmax_pol=q, distance=1.0, min_cell_size=7.0)
            s.set_external_field(np.zeros((n, 3)))
            err.append(np.abs(s.polelec_geomgrad() - gd).max() / np.abs(gd).max())
        assert err[1] <= err[0] / 4.0 and err[2] <= 1.5 * err[1]
    s.terminate()


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("shape", ["cube", "plate", "clump"])
def test_inner_solves(shape, amoeba):
    """Mixed solves large enough for the far-field inner matvec, from nothing and from
    the previous dipoles, before and after a change of coordinates, against the FP64
    solver: a cube, a plate of one layer (most cells empty) and a cube with a few sites
    so far away that it falls into a few leaves (the direct sweep stays).  Both solvers
    stop at an rms of 3e-10 of the preconditioned residual; its inverse operator is
    below 10 here, so that the dipoles agree to an rms of 6e-9."""
    from openmmpol_amd import OMMPSystem
    n = 18001
    spec = chain(n, amoeba, seed=7)
    rng = np.random.default_rng(8)
    if shape == "plate":
        g = np.arange(135)
        p = np.stack(np.meshgrid(g, g, indexing="ij"), axis=-1).reshape(-1, 2)[:n] * 4.0
        spec["cmm"] = np.concatenate([p, np.zeros((n, 1))], axis=1) + rng.uniform(-0.8, 0.8, size=(n, 3))
    elif shape == "clump":
        spec["cmm"][-8:] += 5000.0 * rng.normal(size=(8, 3))
    both = []
    for precision in ("fp64", "mixed"):
        s = OMMPSystem.from_arrays(amoeba, spec["cmm"], spec["q"], spec["pol"], spec["bonds_ri"], spec["bonds_ci"],
                                   pgroup=spec["pgroup"] if amoeba else None)
        s.set_precision(precision)
        s.set_solver_tolerance(3e-10, 500)
        field = np.random.default_rng(9).normal(0.0, 1e-2, size=(2, n, 3))
        got = []
        for scale in (1.0, 1.02):
            if scale != 1.0:
                s.update_coordinates(spec["cmm"] * scale)
            for f in field:
                s.set_external_field(f)
                s.get_polelec_energy()
                got.append(s.ipd.copy())
        both.append(np.array(got))
        s.terminate()
    d = both[0] - both[1]
    assert np.sqrt((d * d).mean(axis=(1, 2, 3))).max() <= 6e-9


def test_kernel_statistics():
    """Mixed solves with far-field inner solves: the class of the direct FP32 sweep
    counts the FP32 residuals (at most one per FP64 step), not the inner products,
    in the first solve and in one enqueued ahead from its iteration counts."""
    n = 13500
    s = _system(n, True)
    s.set_precision("mixed")
    s.set_solver_tolerance(3e-10, 500)
    s.profile_kernels(True)
    field = np.random.default_rng(2).normal(0.0, 1e-2, size=(n, 3))
    for _ in range(2):
        s.kernel_stats(reset=True)
        s.reset_guess()
        s.set_external_field(field)
        outer, inner = s.last_iterations[2:4]
        launches = s.kernel_stats(reset=True)["otf32"][0]
        assert inner >= 2 * outer and 1 <= launches < outer, (launches, outer, inner)
    s.terminate()


@pytest.mark.parametrize("p", [4, 8])
def test_unequal_orders(p):
    """Orders 4 and 8 of the two expansions: the transfer serves the one of order 8,
    the complex kernels and their tables the other; both against trees with an order
    of 9, where the complex kernels serve both (1e-12 as above)."""
    n = 1003
    s = _system(n, True)
    x = np.random.default_rng(3).normal(0.0, 0.05, size=(2, n, 3))
    s.enable_fmm(lmax=12 - p, lmax_pol=p, distance=1.0, min_cell_size=8.0)
    y, e = s.tmatvec(x, kind="fmm")[0], s.e_m2d
    s.enable_fmm(lmax=9, lmax_pol=p, distance=1.0, min_cell_size=8.0)
    want = s.tmatvec(x, kind="fmm")[0]
    assert np.abs(y - want).max() <= 1e-12 * np.abs(want).max()
    s.enable_fmm(lmax=12 - p, lmax_pol=9, distance=1.0, min_cell_size=8.0)
    want = s.e_m2d
    assert np.abs(e - want).max() <= 1e-12 * np.abs(want).max()
    s.terminate()


@pytest.mark.parametrize("amoeba", [True, False])
@pytest.mark.parametrize("n,ncols", [(13500, 1), (13500, 2), (60000, 1), (60000, 2)])
def test_inner_product(n, ncols, amoeba):
    """The FP32 far-field product alone (leaves of 26 and of 117 sites, the latter with
    32 targets a workgroup) against the direct FP64 one.  An inner solve is to reduce
    its residual by 1e-3: 5e-4 of the product's norm asked, and no component further
    off than 20 times the mean error that allows."""
    s = _system(n, amoeba)
    x = np.random.default_rng(4).normal(0.0, 0.05, size=(ncols, n, 3))
    want, _ = s.tmatvec(x, kind="sym64")
    y, _ = s.tmatvec(x, kind="far32")
    assert np.array_equal(s.tmatvec(x, kind="far32")[0], y)
    for m in range(ncols):
        rms = np.sqrt((want[m] ** 2).mean())
        err = np.linalg.norm(y[m] - want[m]) / np.linalg.norm(want[m])
        print(n, ncols, amoeba, f"{err:.1e}")
        assert err <= 5e-4, m
        assert np.abs(y[m] - want[m]).max() <= 20 * 5e-4 * rms, m
    s.terminate()


def _solver(spec, precision, tol, td=None):
    from openmmpol_amd import OMMPSystem
    s = OMMPSystem.from_arrays(True, spec["cmm"], spec["q"], spec["pol"], spec["bonds_ri"], spec["bonds_ci"],
                               pgroup=spec["pgroup"], thole_a=td)
    s.set_precision(precision)
    s.set_solver_tolerance(tol, 500)
    return s


def _solve(s, field):
    """Dipoles, FP64 steps, inner iterations and launches of the direct FP32 sweep."""
    s.kernel_stats(reset=True)
    s.set_external_field(field)
    return (s.ipd.copy(), *s.last_iterations[2:4], s.kernel_stats(reset=True)["otf32"][0])


@pytest.mark.parametrize("shape", ["cube", "plate", "clump"])
def test_inner_path(shape):
    """Which product the inner solves of test_inner_solves' systems run: the far field
    for the cube and the plate (direct FP32 sweeps: at most one residual per FP64 step),
    the direct sweep for the cube that falls into a few leaves.  Iterations: a solve of
    1e-6 in one piece or in two of 1e-3 each, one more per piece."""
    n = 18001
    spec = chain(n, True, seed=7)
    rng = np.random.default_rng(8)
    if shape == "plate":
        g = np.arange(135)
        p = np.stack(np.meshgrid(g, g, indexing="ij"), axis=-1).reshape(-1, 2)[:n] * 4.0
        spec["cmm"] = np.concatenate([p, np.zeros((n, 1))], axis=1) + rng.uniform(-0.8, 0.8, size=(n, 3))
    elif shape == "clump":
        spec["cmm"][-8:] += 5000.0 * rng.normal(size=(8, 3))
    s = _solver(spec, "mixed", 3e-10)
    s.profile_kernels(True)
    field = rng.normal(0.0, 1e-2, size=(n, 3))
    for _ in range(3):
        s.reset_guess()
        _, outer, inner, launches = _solve(s, field)
        print(shape, outer, inner, launches)
        assert outer == 3
        if shape == "clump":
            assert inner <= launches <= inner + 2 * outer
        else:
            assert 1 <= launches < outer
        assert inner <= 30
    s.terminate()


def test_inner_fallback():
    """A geometry that the expansions do not fit: damping factors of 1e-4 damp pairs out
    to 60 bohr, far beyond the 27 leaves of 13 bohr where the product damps them.  The
    direct sweep takes over within the first solve, serves the following ones on this
    geometry, and the far field is tried again on the next (here damped as usual).
    Dipoles against the FP64 solver: T is close to 1 / alpha here, so that two solves to
    an rms of 3e-10 of sqrt(alpha) r differ by sqrt(30) 2 3e-10 = 3.3e-9; 1e-8 asked."""
    n = 18001
    spec = chain(n, True, seed=7)
    spec["pol"][:] = 30.0
    td = np.full(n, 1e-4)
    field = np.random.default_rng(9).normal(0.0, 1e-2, size=(2, n, 3)) + 1e-2
    ref = _solver(spec, "fp64", 3e-10, td)
    s = _solver(spec, "mixed", 3e-10, td)
    s.profile_kernels(True)
    for k, f in enumerate((field[0], field[1], field[0])):
        ref.set_external_field(f)
        got, outer, inner, launches = _solve(s, f)
        print(k, outer, inner, launches)
        assert np.sqrt(((got - ref.ipd) ** 2).mean()) <= 1e-8, k
        assert launches >= 3, k
        if k:
            assert launches >= inner, (k, launches, inner)
    # stretched so far that no pair is damped beyond the leaves: the far field again
    spec["cmm"] = spec["cmm"] * 8.0
    s.update_coordinates(spec["cmm"])
    ref.update_coordinates(spec["cmm"])
    ref.set_external_field(field[0])
    got, outer, inner, launches = _solve(s, field[0])
    print("stretched", outer, inner, launches)
    assert np.sqrt(((got - ref.ipd) ** 2).mean()) <= 1e-8
    assert launches < outer
    ref.terminate()
    s.terminate()


def test_inner_guess_not_finite():
    """A guess that is not finite (written over the dipoles in device memory): the steps
    enqueued ahead come to nothing, the residual after them says so, and the solve starts
    again from nothing with the direct sweep.  Against the solve before it, both to an
    rms of 3e-10 (6e-9 as above)."""
    import ctypes
    n = 18001
    s = _solver(chain(n, True, seed=7), "mixed", 3e-10)
    s.profile_kernels(True)
    field = np.random.default_rng(9).normal(0.0, 1e-2, size=(n, 3))
    want = _solve(s, field)[0]
    bad = np.full((2, n, 3), np.nan)
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipMemcpy(ctypes.c_void_p(s.device_ipd_ptr()), bad.ctypes.data_as(ctypes.c_void_p),
                         ctypes.c_size_t(bad.nbytes), 1) == 0
    got, outer, inner, launches = _solve(s, field)
    print(outer, inner, launches)
    assert np.sqrt(((got - want) ** 2).mean()) <= 6e-9
    assert launches >= 10  # direct inner iterations
    s.terminate()
