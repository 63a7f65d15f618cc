"""Tall-skinny block products at the edges of their tiles: the narrow Gram's
block counts and row remainders, and both tile shapes of Y = U C, against
numpy in 64 bits.

A sum of K products in precision u, in any order, is within (K + 4) u of the
sum of the products' magnitudes."""

import numpy as np
import pytest

from lapy_amd import _lib

pytestmark = pytest.mark.gpu


def _unit(f32):
    return 2.0**-24 if f32 else 2.0**-53


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 130, 1025])
@pytest.mark.parametrize("p,q", [(1, 1), (16, 17), (17, 48), (15, 64), (33, 16), (32, 64), (48, 48), (49, 31), (64, 32)])
def test_narrow_gram(n, p, q, f32):
    rng = np.random.default_rng(n + 100 * p + q)
    U, V = rng.standard_normal((n, 67)), rng.standard_normal((n, 70))
    if f32:
        U, V = U.astype(np.float32).astype(float), V.astype(np.float32).astype(float)
    C, _ = _lib.block_gram(_lib.default_context(), U, V, p, q, f32=f32)
    bound = (n + 4) * _unit(f32) * (np.abs(U[:, :p]).T @ np.abs(V[:, :q]))
    assert np.all(np.abs(C - U[:, :p].T @ V[:, :q]) <= bound)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,p,q,upper,inplace", [
    (1, 3, 16, False, False), (15, 17, 17, False, False), (17, 48, 40, False, False), (33, 16, 129, False, False),
    (33, 33, 33, True, True), (129, 128, 128, True, True), (31, 129, 129, False, True), (513, 200, 200, True, True),
    (24577, 40, 64, False, False), (24577, 40, 80, False, False), (24577, 33, 49, False, False),
    (66001, 72, 72, True, True), (66001, 40, 40, False, True), (99001, 20, 40, False, False),
])
def test_product_tiles(n, p, q, upper, inplace, f32):
    rng = np.random.default_rng(n + p)
    ld = max(p, q) + 3
    U, Cm = rng.standard_normal((n, ld)), rng.standard_normal((p, q))
    if upper:
        Cm = np.triu(Cm)
    if f32:
        U, Cm = U.astype(np.float32).astype(float), Cm.astype(np.float32).astype(float)
    if inplace:
        Y, _ = _lib.block_gemm(_lib.default_context(), None, p, Cm, U, upper=upper, inplace=True, f32=f32)
    else:
        Y, _ = _lib.block_gemm(_lib.default_context(), U, p, Cm, np.zeros((n, ld)), f32=f32)
    bound = (p + 4) * _unit(f32) * (np.abs(U[:, :p]) @ np.abs(Cm))
    assert np.all(np.abs(Y[:, :q] - U[:, :p] @ Cm) <= bound)
    assert np.array_equal(Y[:, q:], U[:, q:] if inplace else np.zeros((n, ld - q)))
