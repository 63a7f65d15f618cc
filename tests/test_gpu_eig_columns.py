"""The eigenvectors' way out of the solver: unpermuted and transposed on the
device in tiles of 64 rows and 32 columns.  Every column is checked against its
own eigenvalue with the host's matrices, so that a value from another row or
column shows: ||A x - l B x|| <= 1e-8 ||B x|| scale, ten times the solver's
tolerance (1e-9 in the same measure) for the rounding of the host's products."""

import numpy as np
import pytest

from lapy_amd import Solver, TriaMesh, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,keep,k", [
    (2, 1.0, 7),     # 162 rows: the dense solver's own columns
    (2, 0.93, 40),   # an odd number of them, past one tile of columns
    (3, 1.0, 31),    # 642 rows: the caller's order, below one tile of columns
    (3, 0.61, 33),   # an odd number of rows, one column into the second tile
    (5, 0.413, 32),  # above 4,096 rows: the locality order undone
    (5, 0.407, 65),  # two full column tiles and one more
])
def test_columns_belong_to_their_eigenvalues(level, keep, k):
    v, t = meshgen.perturbed_sphere(level, np.random.default_rng(k), axes=(1.4, 0.7, 1.0), sigma=0.01)
    if keep < 1.0:
        t = t[(v[:, 2] > np.quantile(v[:, 2], 1 - keep))[t].all(axis=1)]
        used, t = np.unique(t, return_inverse=True)
        v, t = v[used], t.reshape(-1, 3)
    fem = Solver(TriaMesh(v, t))
    lam, x = fem.eigs(k=k)
    assert x.shape == (len(v), k) and x.flags.f_contiguous
    a, b = fem.stiffness, fem.mass
    bx = b @ x
    res = np.linalg.norm(a @ x - bx * lam, axis=0) / np.linalg.norm(bx, axis=0)
    assert np.all(res <= 1e-8 * np.maximum(np.abs(lam), 1e-2 * lam[-1]))
