"""The allocation-free solve when resident launches are refused or give up: the
iteration kernels' result (a handle with event timing), bit for bit, in that
call and, until they are allowed again, in the next ones."""
import ctypes as C

import numpy as np
import pytest

from aphros_amd import _lib as L
from aphros_amd.devmem import DeviceBuffer
from aphros_amd.solver import Poisson

pytestmark = pytest.mark.gpu

DEFAULT = 200000000
SHAPE = (37, 45, 60)


def _system(seed):
    rng = np.random.default_rng(seed)
    k = [rng.uniform(0.5, 1.5, SHAPE) for _ in range(3)]
    E = np.empty(SHAPE + (8,))
    for d, (kf, a) in enumerate(zip(k, (2, 1, 0))):
        E[..., 1 + 2 * d] = -kf
        E[..., 2 + 2 * d] = -np.roll(kf, -1, a)
    E[..., 0] = 1.0 - E[..., 1:7].sum(-1)
    E[..., 7] = rng.standard_normal(SHAPE)
    return E


@pytest.fixture
def wait():
    def set_(ticks):
        L.check(L.lib().aphpois_noalloc_set_resident_wait(0, ticks))
    yield set_
    set_(0)


@pytest.mark.parametrize("maxiter", [0, 40])
@pytest.mark.parametrize("ticks", [-1, -2 ** 63])
@pytest.mark.parametrize("method", [L.CONJUGATE, L.JACOBI])
def test_fallback_and_its_memory(method, ticks, maxiter, wait):
    E = _system(1)
    e_dev, x_dev = DeviceBuffer(E.nbytes), DeviceBuffer(E.nbytes // 8)
    e_dev.from_host(E)
    d = L.Desc()
    L.lib().aphpois_desc_default(C.byref(d))
    d.nz, d.ny, d.nx = SHAPE
    d.method, d.resmode, d.tol, d.miniter, d.maxiter, d.h3 = method, L.RES_L2, 0.0, 0, maxiter, 1.0

    def solve():
        info = L.Info()
        L.check(L.lib().aphpois_solve_device_noalloc(C.byref(d), e_dev.ptr, None, x_dev.ptr, None,
                                                     C.byref(info)))
        assert info.iter == maxiter + 1
        return x_dev.to_host(np.empty(SHAPE))
    resident = solve()
    s = Poisson(SHAPE, method=method, resmode=L.RES_L2, tol=0.0, miniter=0, maxiter=maxiter, h3=1.0)
    s.set_system(E)
    s.set_profiling(True)
    launched, _ = s.solve(None)
    s.close()
    wait(ticks)
    x = solve()
    # (workgroups that met all the same count, and nothing is remembered)
    kept = ticks == -1 and np.array_equal(x, resident)
    assert kept or np.array_equal(x, launched)
    if not kept:
        wait(DEFAULT)
        assert np.array_equal(solve(), launched)
    wait(0)
    assert np.array_equal(solve(), resident)
    e_dev.free()
    x_dev.free()


def test_wait_of_an_unknown_device():
    assert L.lib().aphpois_noalloc_set_resident_wait(-1, 0) == L.EINVAL
    assert L.lib().aphpois_noalloc_set_resident_wait(1 << 20, 0) == L.EINVAL
