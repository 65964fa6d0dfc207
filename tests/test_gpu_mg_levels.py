"""One multigrid cycle against the oracle's at the sizes where a level changes
its kernels: small fused levels and their workgroup sizes, short and long rows, partial row tiles, with and without a mass
term and W levels."""
import numpy as np
import pytest

from aphros_amd import _lib as L
from aphros_amd.batch import Batch
from aphros_amd.solver import Poisson
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {L.FP64: 1e-12, L.MIXED: 1e-4}  # rounding; bfloat16 coefficients restated


def _system(shape, seed, mass):
    rng = np.random.default_rng(seed)
    rho = np.where(rng.random(shape) < 0.2, 100.0, 1.0)
    f = rng.standard_normal(shape)
    e = O.assemble(rho, f - f.mean())
    if mass:
        e[..., 0] *= 1.0 + 1e-3 * rng.random(shape)
    return np.ascontiguousarray(e)


def _cycle_error(shape, precision, w, mass, seed=1):
    e = _system(shape, seed, mass)
    s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                maxiter=2000, precond=L.PRECOND_MG, mg_w=w)
    s.set_system(e)
    r = np.random.default_rng(seed + 1).standard_normal(shape)
    if not mass:
        r -= r.mean()
    z = s.precond_apply(r)
    x, info = s.solve(None)
    s.close()
    assert info["converged"] == 1 and O.true_relres(e, x) <= 1e-8 * (1 + 1e-6)
    zo, nlev = O.mg_apply(e, r, bf16=precision == L.MIXED, w=w)
    err = np.abs(z - zo).max() / np.abs(zo).max()
    print(shape, precision, w, mass, "levels", nlev, "iter", info["iter"], "err", err, flush=True)
    return err


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("precision,shape,w", [
    (L.FP64, (128, 64, 64), 0),       # 2^19 cells
    (L.FP64, (64, 256, 32), 1),       # rows of 16 threads
    (L.FP64, (64, 96, 96), 2),        # rows of 48 threads, a partial row tile
    (L.FP64, (8, 256, 256), 1),       # rows of 128 threads, 8 planes
    (L.MIXED, (192, 128, 128), 0),    # 3 * 2^20 cells
    (L.MIXED, (768, 128, 32), 1),     # rows of 8 threads
    (L.MIXED, (128, 160, 160), 2),    # rows of 40 threads, a partial row tile
    (L.MIXED, (16, 768, 256), 1),     # rows of 64 threads, 16 planes
])
def test_smallest_fused_levels(precision, shape, w, mass):
    assert _cycle_error(shape, precision, w, mass) <= TOL[precision]


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("precision,shape,w", [
    (L.MIXED, (64, 64, 96), 0),       # 3 * 2^17 cells, 256 threads
    (L.MIXED, (40, 136, 80), 0),      # 12 rows of 20 threads, a partial row tile
    (L.MIXED, (96, 80, 64), 1),       # 16 rows of 16 threads, partial in y and z
    (L.MIXED, (24, 128, 128), 0),     # 8 rows of 32 threads, 256 threads
    (L.MIXED, (24, 128, 144), 0),     # 36 threads a row: 512 threads
    (L.MIXED, (8, 200, 256), 0),      # 64 threads a row, 8 planes, partial
    (L.MIXED, (24, 64, 272), 0),      # 68 threads a row: 1024 threads
    (L.MIXED, (128, 256, 256), 1),    # 2^23 cells, levels of 1024 and 256 threads
    (L.FP64, (16, 16, 16), 0),        # the smallest fused level
    (L.FP64, (8, 8, 66), 0),          # 33 threads a row: 512 threads, 10 rows
    (L.FP64, (8, 34, 64), 0),         # 8 rows of 32 threads, partial, 8 planes
    (L.FP64, (8, 32, 136), 0),        # 68 threads a row: 1024 threads
    (L.FP64, (40, 48, 20), 1),        # 24 rows of 10 threads
])
def test_fused_workgroup_sizes(precision, shape, w, mass):
    assert _cycle_error(shape, precision, w, mass) <= TOL[precision]


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("precision", [L.FP64, L.MIXED])
@pytest.mark.parametrize("shape", [
    (8, 8, 8),        # the bottom is one wavefront's (4^3, 2^3)
    (6, 6, 6),        # one coarsest level of 27 cells
    (10, 10, 10),     # one coarsest level of 125 cells, all threads
    (20, 20, 20),     # 10^3 above a coarsest level of 5^3
    (24, 24, 24),     # 12^3, 6^3 and a wavefront's 3^3
    (28, 28, 28),     # 14^3 (rows of 14), coarsest 7^3
    (32, 24, 40),     # 3840, 480 and 60 cells
    (32, 32, 32),     # 4096, 512, 64 and 8 cells
    (4, 4, 2048),     # 2 x 2 x 1024 cells above 1 x 1 x 512
    (30, 30, 30),     # a coarsest level of 3375 cells
    (64, 64, 128),    # 2^19 cells: the largest level in tiles
    (36, 44, 52),     # partial tiles on every side
])
def test_bottom_levels(shape, precision, mass):
    assert _cycle_error(shape, precision, 0, mass) <= TOL[precision]


def test_largest_coarsest_level():
    """19^3 cells on the coarsest of two levels, more than the threads hold:
    FP32 engines only, beyond what the oracle's cycle takes."""
    shape = (38, 38, 38)
    e = _system(shape, 3, False)
    s = Poisson(shape, method=L.PCG, precision=L.MIXED, resmode=L.RES_REL_TRUE, tol=1e-8,
                maxiter=2000, precond=L.PRECOND_MG)
    s.set_system(e)
    x, info = s.solve(None)
    s.close()
    assert info["converged"] == 1 and O.true_relres(e, x) <= 1e-8 * (1 + 1e-6)


@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
def test_reductions_at_the_size_line(precision):
    """2^23 cells (reductions finished by the kernels that need them), 5/4 as
    many (by kernels of their own), both in one batch with a small system:
    each as alone, bit for bit, also from a guess and cut short by maxiter."""
    shapes = [(128, 256, 256), (160, 256, 256), (16, 24, 20)]
    es = [_system(s, 5 + i, i == 2) for i, s in enumerate(shapes)]
    b = Batch(precision=precision, tol=1e-8, maxiter=2000, precond=L.PRECOND_MG,
              mg_w=L.MG_W_AUTO)
    slots = [b.add(e) for e in es]
    b.solve()
    for e, shape, slot in zip(es, shapes, slots):
        xb, ib = b.get(slot)
        s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                    maxiter=2000, precond=L.PRECOND_MG)
        s.set_system(e)
        x, info = s.solve(None)
        assert ib["converged"] == info["converged"] == 1 and ib["iter"] == info["iter"]
        assert np.array_equal(x, xb) and O.true_relres(e, x) <= 1e-8 * (1 + 1e-6)
        x2, warm = s.solve(x + 3.0 if shape[0] != 16 else x)
        assert warm["converged"] == 1 and warm["iter"] <= 2
        assert O.true_relres(e, x2) <= 1e-8 * (1 + 1e-6)
        s.close()
        s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                    maxiter=3, precond=L.PRECOND_MG)
        s.set_system(e)
        x3, cut = s.solve(None)
        s.close()
        assert cut["converged"] == 0 and cut["iter"] == 4
        assert abs(O.true_relres(e, x3) / cut["true_relres"] - 1) <= 1e-6
    b.close()


@pytest.mark.parametrize("precond", [L.PRECOND_MG, L.PRECOND_JACOBI])
@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
@pytest.mark.parametrize("shape", [
    (16, 40, 288),    # 72 / 144 columns
    (48, 40, 160),    # 40 / 80 columns
    (16, 24, 104),    # 26 / 52 columns
    (64, 128, 288),   # beyond the resident solves
    (80, 96, 336),    # 84 / 168 columns
])
def test_row_tiles_that_are_no_power_of_two(shape, precision, precond):
    e = _system(shape, 9, False)
    s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                maxiter=5000, precond=precond)
    s.set_system(e)
    x, info = s.solve(None)
    s.close()
    assert info["converged"] == 1
    assert abs(O.true_relres(e, x) / info["true_relres"] - 1) <= 1e-6


@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
def test_new_systems_in_one_slot(precision):
    """A time loop's systems, some with a mass term, one after the other in a
    solver: each as in a solver of its own, bit for bit."""
    shape = (24, 40, 48)

    def solver():
        return Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                       maxiter=2000, precond=L.PRECOND_MG)
    loop = solver()
    for seed, mass in ((1, False), (2, False), (3, True), (4, False), (5, True)):
        e = _system(shape, seed, mass)
        loop.set_system(e)
        x, info = loop.solve(None)
        own = solver()
        own.set_system(e)
        xo, io = own.solve(None)
        own.close()
        assert info["converged"] == 1 and info["iter"] == io["iter"]
        assert np.array_equal(x, xo) and O.true_relres(e, x) <= 1e-8 * (1 + 1e-6)
    loop.close()


@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
@pytest.mark.parametrize("shape", [(16, 24, 20), (64, 96, 80), (160, 256, 256)])
def test_breakdown_ends_the_solve(shape, precision):
    """b = 0 and more iterations asked for: (p, q) = 0 in the first, which ends the
    solve and leaves x as it was, at sizes of either form of the reductions; the
    solver then solves as a new one, bit for bit."""
    e = _system(shape, 7, False)

    def solver():
        s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                    miniter=3, maxiter=2000, precond=L.PRECOND_MG)
        s.set_system(e)
        return s
    s = solver()
    for _ in range(3):
        s.set_rhs(np.zeros(shape))
        x, info = s.solve(None)
        assert info["status"] == L.ENUMERIC and info["iter"] == 0 and info["converged"] == 0
        assert not x.any()
        s.set_rhs(e[..., 7])
        x, info = s.solve(None)
        assert info["status"] == 0 and info["converged"] == 1
    s.close()
    own = solver()
    xo, io = own.solve(None)
    own.close()
    assert info["iter"] == io["iter"] and np.array_equal(x, xo)


@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
@pytest.mark.parametrize("shape", [
    (16, 40, 288),    # 72 / 144 columns
    (48, 40, 160),    # 40 / 80 columns
    (16, 24, 104),    # 26 / 52 columns
    (20, 18, 77),     # 77 columns of one cell
])
def test_row_tiles_of_the_jacobi_scaled_operator(shape, precision):
    """The same tiles in the Jacobi-scaled operator and update, which systems of
    these sizes launch only with event timing on: the resident solve's iterations
    and solution."""
    e = _system(shape, 9, True)
    got = []
    for timed in (False, True):
        s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-10,
                    maxiter=5000, precond=L.PRECOND_JACOBI)
        s.set_system(e)
        s.set_profiling(timed)
        x, info = s.solve(None)
        s.close()
        assert info["converged"] == 1
        assert O.true_relres(e, x) <= 1e-10 * (1 + 1e-6)
        got.append((x, info["iter"]))
    (x, i), (xk, ik) = got
    err = np.linalg.norm((x - xk).ravel()) / np.linalg.norm(x.ravel())
    print(shape, precision, i, ik, err, flush=True)
    assert abs(i - ik) <= max(1, i // 50)


@pytest.mark.parametrize("lx", [64, 128, 256])
@pytest.mark.parametrize("precision,shape", [
    (L.FP64, (8, 16, 264)),     # 132 columns: too long for the fused kernels
    (L.MIXED, (16, 16, 98)),    # 49 columns of two cells
])
def test_tile_override_on_a_swept_level(precision, shape, lx):
    """Rows of a tile as long as the workgroup: the restriction, which sums row
    pairs inside a workgroup, still has two rows."""
    e = _system(shape, 11, False)
    s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                maxiter=2000, precond=L.PRECOND_MG, mg_w=0)
    s.set_system(e)
    s.set_tile(lx=lx)
    r = np.random.default_rng(12).standard_normal(shape)
    r -= r.mean()
    z = s.precond_apply(r)
    s.close()
    zo, nlev = O.mg_apply(e, r, bf16=precision == L.MIXED, w=0)
    assert np.abs(z - zo).max() <= TOL[precision] * np.abs(zo).max()
