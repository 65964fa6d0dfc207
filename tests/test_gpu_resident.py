"""Resident solves (small systems of CONJUGATE, JACOBI and Jacobi-scaled PCG
whose iterations run in one cooperative launch): sizes at the edges of every
kernel instance (columns per thread x cells per column: 1x1, 1x2, 1x4, 1x8,
2x8), ragged boxes, edges of 1, solves of more than one launch (512
iterations), against the oracle and against the iteration kernels (event
timing on).

Systems: random symmetric face coefficients in [0.5, 1.5] plus a mass term of
1, so the spectrum of A lies in [1, 19] and an error in x is at most 19 times
the relative residual (2-norms)."""
import ctypes as C

import numpy as np
import pytest

from aphros_amd import _lib as L
from aphros_amd.devmem import hip
from aphros_amd.solver import Poisson
from oracle import oracle as O

pytestmark = pytest.mark.gpu

COND = 19.0
# nz, ny, nx
SHAPES = [
    (1, 1, 1), (1, 1, 7), (5, 7, 1), (2, 1, 9),      # edges of 1
    (16, 16, 16),                                    # one column, one cell
    (32, 33, 31), (52, 45, 60),                      # two and four cells
    (93, 75, 101),                                   # eight cells, ragged boxes
    (121, 117, 127),                                 # two columns of eight
    (16, 8, 700),                                    # rows longer than a workgroup
    (128, 128, 128),                                 # the largest
]


def _system(shape, seed, sign=1.0):
    rng = np.random.default_rng(seed)
    k = [rng.uniform(0.5, 1.5, shape) for _ in range(3)]  # lower faces x, y, z
    E = np.empty(shape + (8,))
    for d, (kf, a) in enumerate(zip(k, (2, 1, 0))):
        E[..., 1 + 2 * d] = -kf
        E[..., 2 + 2 * d] = -np.roll(kf, -1, a)
    E[..., 0] = 1.0 - E[..., 1:7].sum(-1)
    E[..., 7] = rng.standard_normal(shape)
    return np.ascontiguousarray(sign * E)


def _err(x, y):
    return np.linalg.norm((x - y).ravel()) / np.linalg.norm(y.ravel())


@pytest.mark.parametrize("shape", SHAPES)
def test_jacobi_bit_for_bit(shape):
    E = _system(shape, 1)
    sweeps = 600 if np.prod(shape) <= 40000 else 5  # > 512: a second launch
    s = Poisson(shape, method=L.JACOBI, resmode=L.RES_L2, tol=0.0, miniter=0,
                maxiter=sweeps - 1, h3=1.0)
    s.set_system(E)
    x, info = s.solve(None)
    s.close()
    xo, ito, reso, _ = O.jacobi(E, tol=0.0, miniter=0, maxiter=sweeps - 1)
    print(shape, info["iter"], ito, flush=True)
    assert info["iter"] == ito == sweeps
    assert np.array_equal(x, xo) and info["residual"] == reso


@pytest.mark.parametrize("shape", SHAPES)
def test_conjugate(shape):
    """8 iterations and their continuation from there; 100 times the rounding
    of a sum as the bound (each iterate's error is a few roundings times the
    condition number)."""
    E = _system(shape, 2)
    s = Poisson(shape, method=L.CONJUGATE, resmode=L.RES_MAX, tol=0.0, miniter=0, maxiter=7,
                h3=1.0)
    s.set_system(E)
    x, info = s.solve(None)
    xo, ito, reso, _ = O.conjugate(E, 1.0, tol=0.0, miniter=0, maxiter=7, maxnorm=True)
    print(shape, info["iter"], ito, _err(x, xo), flush=True)
    assert info["iter"] == ito
    n_exact = int(np.prod(shape))
    if n_exact > 8:  # (a smaller system has converged before; 0/0 follows)
        assert _err(x, xo) <= 100 * COND * 2.3e-16 * 8
        assert abs(info["residual"] - reso) <= 1e-9 * abs(reso)
        y0, _ = s.solve(x)
        yo, _, _, _ = O.conjugate(E, 1.0, x0=xo, tol=0.0, miniter=0, maxiter=7, maxnorm=True)
        assert _err(y0, yo) <= 100 * COND * 2.3e-16 * 8
    s.close()


@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_pcg(shape, precision, sign):
    tol = 1e-10
    E = _system(shape, 3, sign)
    s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=tol,
                maxiter=5000, precond=L.PRECOND_JACOBI)
    s.set_system(E)
    x, info = s.solve(None)
    assert info["converged"] == 1 and info["status"] == 0
    assert O.true_relres(E, x) <= tol * (1 + 1e-6)
    # warm start from the solution of another right-hand side
    E2 = E.copy()
    E2[..., 7] *= 1.01
    s.set_rhs(E2[..., 7])
    y, iw = s.solve(x)
    assert iw["converged"] == 1 and iw["iter"] <= info["iter"]
    assert _err(y, 1.01 * x) <= 2 * COND * tol
    s.set_rhs(E[..., 7])
    # the iteration kernels
    s.set_profiling(True)
    xk, ik = s.solve(None)
    s.close()
    print(shape, precision, info["iter"], ik["iter"], _err(x, xk), flush=True)
    assert abs(info["iter"] - ik["iter"]) <= 1
    assert _err(x, xk) <= 2 * COND * tol


def test_pcg_without_a_mass_term_reaches_maxiter():
    """The zero row sums' operator; the limit of iterations ends the solve in
    the middle of a launch, as the iteration kernels end it."""
    E = _system((20, 24, 28), 4)
    E[..., 0] = -E[..., 1:7].sum(-1)
    E[..., 7] -= E[..., 7].mean()
    got = []
    for prof in (False, True):
        s = Poisson((20, 24, 28), method=L.PCG, precision=L.FP64, resmode=L.RES_REL_TRUE,
                    tol=1e-13, maxiter=40, precond=L.PRECOND_JACOBI)
        s.set_system(E)
        s.set_profiling(prof)
        got.append(s.solve(None))
        s.close()
    (x, i), (xk, ik) = got
    assert i["iter"] == ik["iter"] == 41 and i["converged"] == ik["converged"] == 0
    assert i["refinements"] == ik["refinements"]
    assert _err(x, xk) <= 1e-9


@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI, L.PCG])
def test_workgroups_that_do_not_meet(method):
    """A resident launch whose workgroups give up waiting at once changes
    nothing: the solve is then that of the iteration kernels, bit for bit."""
    shape = (40, 36, 44)
    E = _system(shape, 5)
    got = []
    for wait in (False, True):
        kw = dict(resmode=L.RES_REL_TRUE, tol=1e-9) if method == L.PCG else \
            dict(resmode=L.RES_L2, tol=1e-6)
        s = Poisson(shape, method=method, miniter=0, maxiter=2000, h3=1.0, **kw)
        s.set_system(E)
        if wait:
            s.set_resident_wait(-1)
        else:
            s.set_profiling(True)
        got.append([s.solve(None), s.solve(None)])
        s.close()
    for (x, i), (xk, ik) in zip(*got):
        assert i["converged"] == ik["converged"] == 1 and i["iter"] == ik["iter"]
        assert np.array_equal(x, xk)


def test_served_large_and_small_lanes():
    """One lane's resident launches beside the other lane's captured graph."""
    from aphros_amd.serve import Server
    big, small = _system((132, 128, 128), 6), _system((48, 48, 48), 7)
    srv = Server(precision=L.MIXED, tol=1e-8, precond=L.PRECOND_JACOBI)
    ids = [srv.submit(e, nsteps=3, seed=k, want_x=True)
           for k, e in enumerate((small, big, small, big, small))]
    res = [srv.wait(i, timeout=60) for i in ids]
    alone = srv.wait(srv.submit(small, nsteps=3, seed=2, want_x=True), timeout=60)
    srv.close()
    assert all(r["status"] == 0 and r["last_relres"] <= 1e-8 for r in res)
    assert np.array_equal(res[2]["x"], alone["x"])


@pytest.mark.parametrize("shape", [(33, 35, 37), (52, 45, 60), (93, 75, 101), (121, 117, 127)])
@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI, L.PCG])
def test_early_row_loads_that_lapse(method, shape):
    """The wait for the neighbours' rows gives up at once while the workgroups do
    meet: the rows are then loaded behind the sums, so the solve is the same, bit
    for bit (JACOBI: the oracle's)."""
    E = _system(shape, 8)
    got = []
    for early in (None, -1):
        if method == L.JACOBI:
            kw = dict(resmode=L.RES_L2, tol=0.0, maxiter=11)
        elif method == L.CONJUGATE:
            kw = dict(resmode=L.RES_L2, tol=1e-6, maxiter=2000)
        else:
            kw = dict(resmode=L.RES_REL_TRUE, tol=1e-9, maxiter=2000)
        s = Poisson(shape, method=method, miniter=0, h3=1.0, **kw)
        s.set_system(E)
        if early is not None:
            s.set_resident_wait(200000000, early)
        got.append(s.solve(None))
        s.close()
    (x, i), (y, j) = got
    assert i["iter"] == j["iter"] and np.array_equal(x, y)
    if method == L.JACOBI:
        xo, ito, _, _ = O.jacobi(E, tol=0.0, miniter=0, maxiter=11)
        assert ito == j["iter"] and np.array_equal(y, xo)
    else:
        assert j["converged"] == 1


@pytest.mark.parametrize("shape", [(33, 35, 37), (93, 75, 101)])
@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI, L.PCG])
def test_wait_that_lapses_in_the_last_gather(method, shape):
    """One iteration, whose last gather some workgroups may find complete while
    others give up at once: the launch counts for all of them or for none, so
    every solve is that of the resident or that of the iteration kernels, bit for
    bit (JACOBI: the oracle's)."""
    E = _system(shape, 9)
    kw = dict(resmode=L.RES_REL_TRUE, tol=1e-14) if method == L.PCG else \
        dict(resmode=L.RES_L2, tol=0.0)

    def solve(setup):
        s = Poisson(shape, method=method, miniter=0, maxiter=0, h3=1.0, **kw)
        s.set_system(E)
        setup(s)
        x, info = s.solve(None)
        s.close()
        assert info["iter"] == 1 and info["converged"] == 0
        return x
    whole = [solve(lambda s: None), solve(lambda s: s.set_profiling(True))]
    for _ in range(12):
        x = solve(lambda s: s.set_resident_wait(-1))
        assert any(np.array_equal(x, w) for w in whole)
    if method == L.JACOBI:
        xo, ito, _, _ = O.jacobi(E, tol=0.0, miniter=0, maxiter=0)
        assert ito == 1 and np.array_equal(x, xo)


@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI, L.PCG])
def test_refused_launch(method):
    """A resident launch that the runtime refuses is answered by the iteration
    kernels, in this solve and the next."""
    shape = (40, 36, 44)
    E = _system(shape, 10)
    kw = dict(resmode=L.RES_REL_TRUE, tol=1e-9) if method == L.PCG else \
        dict(resmode=L.RES_L2, tol=1e-6)
    got = []
    for setup in (lambda s: s.set_profiling(True), lambda s: s.set_resident_wait(-2 ** 63)):
        s = Poisson(shape, method=method, miniter=0, maxiter=2000, h3=1.0, **kw)
        s.set_system(E)
        setup(s)
        got.append([s.solve(None), s.solve(None)])
        s.close()
    for (xk, ik), (x, i) in zip(*got):
        assert i["converged"] == ik["converged"] == 1 and i["iter"] == ik["iter"]
        assert np.array_equal(x, xk)


@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI, L.PCG])
def test_device_memory_is_what_the_budget_counts(method):
    """A 128^3 solver holds the bytes it reports (and a budget of these lets it
    solve), up to scratch that does not grow with the system."""
    shape = (128, 128, 128)
    E = _system(shape, 11)
    kw = dict(resmode=L.RES_REL_TRUE, tol=1e-6) if method == L.PCG else \
        dict(resmode=L.RES_L2, tol=0.0)

    def unused():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    def solve(budget):
        free = unused()
        s = Poisson(shape, method=method, miniter=0, maxiter=3, h3=1.0, mem_budget=budget, **kw)
        s.set_system(E)
        x, info = s.solve(None)
        used, told = free - unused(), s.device_bytes()
        s.close()
        return x, used, told
    solve(0)  # (code objects and the like)
    x, used, told = solve(0)
    print(method, used, told, flush=True)
    assert used <= told + (14 << 20)
    y, _, again = solve(told)
    assert again == told and np.array_equal(x, y)


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("precision", [L.MIXED, L.FP64])
def test_launches_with_several_workgroups_per_unit(precision, mass):
    """A batch of more systems than compute units have workgroups for, of one to
    four cells per thread: each as alone, bit for bit."""
    from aphros_amd.batch import Batch
    shapes = [(16, 16, 16), (32, 32, 32), (33, 40, 48), (64, 64, 64)]
    es = []
    for k, shape in enumerate(shapes):
        e = _system(shape, 20 + k)
        if not mass:
            e[..., 0] = -e[..., 1:7].sum(-1)
            e[..., 7] -= e[..., 7].mean()
        es.append(e)
    b = Batch(precision=precision, tol=1e-8, maxiter=5000, precond=L.PRECOND_JACOBI)
    slots = [(b.add(es[k]), k, c) for c in range(9) for k in range(len(es))]
    for sl, k, c in slots:  # nine right-hand sides per system
        b.set_rhs(sl, np.roll(es[k][..., 7], c, axis=0), np.zeros(shapes[k]))
    b.solve()
    for k, shape in enumerate(shapes):
        s = Poisson(shape, method=L.PCG, precision=precision, resmode=L.RES_REL_TRUE, tol=1e-8,
                    maxiter=5000, precond=L.PRECOND_JACOBI)
        s.set_system(es[k])
        for sl, kk, c in slots:
            if kk != k:
                continue
            s.set_rhs(np.roll(es[k][..., 7], c, axis=0))
            x, info = s.solve(None)
            xb, ib = b.get(sl)
            assert info["converged"] == ib["converged"] == 1 and info["iter"] == ib["iter"]
            assert np.array_equal(x, xb)
        s.close()
    b.close()


@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI, L.PCG])
def test_guess_with_wide_strides(method):
    """A guess whose strided range exceeds what set_system staged (the buffer moves
    between the table's set-up and the solve), in place: as the dense guess, bit
    for bit."""
    shape = (6, 5, 7)
    nz, ny, nx = shape
    E = _system(shape, 12)
    kw = dict(resmode=L.RES_REL_TRUE, tol=1e-10) if method == L.PCG else \
        dict(resmode=L.RES_L2, tol=0.0, maxiter=6)
    s = Poisson(shape, method=method, miniter=0, h3=1.0, **kw)
    s.set_system(E)
    x0 = np.random.default_rng(1).standard_normal(shape)
    s.solve(None)
    ly, lz, start = 130, 2600, 55
    wide = np.full(start + nz * lz, 7.0)
    inner = np.lib.stride_tricks.as_strided(wide[start:], shape, (8 * lz, 8 * ly, 8))
    inner[...] = x0
    info = L.Info()
    L.check(L.lib().aphpois_solve(s.h, L.dptr(wide), L.dptr(wide), start, ly, lz, C.byref(info)))
    x, dense = s.solve(x0)
    s.close()
    assert info.iter == dense["iter"] and np.array_equal(inner, x)
    inner[...] = 7.0
    assert np.all(wide == 7.0)
