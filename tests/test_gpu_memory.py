"""The memory that a context keeps between calls, and solves on a device with
little left: what fitted without the kept memory and the multigrid hierarchy
still runs."""

import ctypes as C

import numpy as np
import pytest
from scipy import sparse

from lapy_amd import Solver, TriaMesh, _lib, meshgen

pytestmark = pytest.mark.gpu

MB = 1 << 20


class _Hip:
    def __init__(self):
        _lib.lib()  # the library first: the HIP runtime it links is the one loaded below
        self.h = C.CDLL("/opt/rocm/lib/libamdhip64.so.7")
        self.h.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.h.hipFree.argtypes = [C.c_void_p]
        self.h.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
        self.held = []

    def free(self):
        f, t = C.c_size_t(), C.c_size_t()
        assert self.h.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    def leave(self, nbytes):
        """Take device memory until nbytes are left."""
        while self.free() > nbytes + 2 * MB:
            p = C.c_void_p()
            take = min(self.free() - nbytes, 32 << 30) // MB * MB
            assert self.h.hipMalloc(C.byref(p), take) == 0
            self.held.append(p)

    def close(self):
        for p in self.held:
            self.h.hipFree(p)
        self.held = []


@pytest.fixture
def hip():
    h = _Hip()
    yield h
    h.close()


def _fem():
    return Solver(TriaMesh(*meshgen.perturbed_sphere(5, np.random.default_rng(2), sigma=0.02)), lump=True)


def test_trim_gives_the_kept_memory_back(hip):
    ctx = _lib.default_context()
    fem = _fem()
    lam, x = fem.eigs(k=10)
    before = hip.free()
    ctx.trim()
    assert hip.free() >= before + 256 * MB  # the eigensolver's work memory starts there
    ctx.trim()  # nothing left to give
    again, y = fem.eigs(k=10)
    assert np.array_equal(again, lam) and np.array_equal(y, x)


def test_other_calls_get_the_kept_memory(hip):
    """An allocation of another entry point that fits only without it."""
    ctx = _lib.default_context()
    fem = _fem()
    fem.eigs(k=10)
    hip.leave(96 * MB)
    p, q, n = 8, 8, 2 * MB  # two blocks of 128 MiB
    U = np.random.default_rng(0).standard_normal((n, p))
    c, _ = _lib.block_gram(ctx, U, U, p, q, sym=True)
    hip.close()
    assert np.allclose(c, U.T @ U, rtol=1e-12, atol=1e-9 * n**0.5)


def test_linear_solve_with_little_memory(hip):
    """800 columns of 10,242 rows: six blocks of 66 MB for Jacobi's solve; the
    cycle has more than four of its own."""
    ctx = _lib.default_context()
    fem = _fem()
    a = sparse.csr_matrix(fem.stiffness)
    n, m = a.shape[0], 800
    b = np.random.default_rng(1).standard_normal((n, m))
    b -= b.mean(axis=0)
    _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b[:, :2], rtol=1e-12)  # the order, built once
    ctx.trim()
    hip.leave(560 * MB)
    x, st = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, rtol=1e-12)
    hip.close()
    print("iterations", st.iterations)
    assert st.iterations > 200  # Jacobi
    r = b - a @ x
    assert np.all(np.linalg.norm(r, axis=0) <= 1e-11 * np.linalg.norm(b, axis=0))
