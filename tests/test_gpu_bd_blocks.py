"""The Cholesky factor at the edges of panels and outer blocks against the FP64
factor, its pivot check, and the step's products and forces at the edges of
their blocks."""
import ctypes

import numpy as np
import pytest

import oracle
from test_zz_no_alloc import D2H, H2D, _hip
from tis_amd.bdhi import bead_spring_chain
from tis_amd.engine import BDEngine, load_library


def _factor(a):
    """(return code, failing pivot + 1, factor) of the symmetric matrix a."""
    hip, n, nbytes = _hip(), len(a), a.nbytes
    fn = load_library().tis_bdhi_factor_noalloc
    fn.restype = ctypes.c_int32
    fn.argtypes = [ctypes.c_int32, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32, ctypes.c_void_p, ctypes.c_void_p]
    D, L, info = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_int32(-1)
    assert hip.hipMalloc(ctypes.byref(D), nbytes) == 0 and hip.hipMalloc(ctypes.byref(L), nbytes) == 0
    try:
        assert hip.hipMemcpy(D, a.ctypes.data, nbytes, H2D) == 0
        rc = fn(0, D, L, n, None, ctypes.byref(info))
        assert hip.hipDeviceSynchronize() == 0
        out = np.zeros((n, n), order="F")
        assert hip.hipMemcpy(out.ctypes.data, L, nbytes, D2H) == 0
    finally:
        hip.hipFree(D)
        hip.hipFree(L)
    return rc, info.value, out


def _spd(n):
    g = np.random.default_rng(n).standard_normal((n, n))
    return g @ g.T / n + np.eye(n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 16, 63, 64, 65, 80, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 511, 577])
def test_factor_sizes(n):
    a = _spd(n)
    print(f"[factor] n={n}", flush=True)
    rc, info, L = _factor(a)
    assert rc == 0 and info == 0
    l64 = np.linalg.cholesky(a)
    err = np.abs(L - l64).max() / np.abs(l64).max()
    # one panel is FP64 throughout; further ones take products in FP32
    assert err <= (1e-13 if n <= 64 else 2e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("p", [0, 15, 16, 47, 63, 64, 100, 129])
def test_pivot_check(p):
    a = _spd(130)
    a[p, p] = -1.0
    print(f"[pivot] {p}", flush=True)
    rc, info, _ = _factor(a)
    assert rc != 0 and info == p + 1


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 3, 21, 22, 64, 65, 66, 130])
def test_forces_and_step(n):
    """Lanes of one bead's pairs (64 and more), rows and columns of the step's
    products at the edges of their blocks; bounds as for the chains of the
    step and force tests."""
    s, x = bead_spring_chain(n, seed=n)
    print(f"[bd] n={n}", flush=True)
    e = BDEngine(s, key=9, seed=11)
    e.set_coords(x)
    f, fo = e.forces(), oracle.bd_forces(s, x)
    assert np.abs(f - fo).max() <= 1e-12 * max(1.0, np.abs(fo).max())
    e.steps(3, tstep=0.05, refactor_every=1, step0=100)
    xo = oracle.bdhi_run(s, x, 3, tstep=0.05, refactor_every=1, seed=11, key=9, step0=100)
    assert np.abs(e.coords() - xo).max() <= 1e-5
    e.close()
