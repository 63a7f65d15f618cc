"""Sparsity patterns of rows with few and very many elements, and the buffered
pairwise sums behind the mean edge length, against the CPU oracle."""

import numpy as np
import pytest

from lapy_amd import Solver, TetMesh, TriaMesh
from oracle import fem

pytestmark = pytest.mark.gpu


def _fan(valence):
    a = 2 * np.pi * np.arange(valence) / valence
    v = np.vstack([[0.0, 0.0, 0.3], np.c_[np.cos(a), np.sin(a), 0.1 * np.cos(3 * a)]])
    i = np.arange(valence)
    return v, np.c_[np.zeros(valence, int), 1 + i, 1 + (i + 1) % valence]


def _spindle(valence):
    """Tets around one edge."""
    v, t = _fan(valence)
    v = np.vstack([v, [[0.0, 0.0, 2.0]]])
    return v, np.c_[t, np.full(valence, valence + 1)]


# 8 and 16 lanes a row, two records each in registers: 16 triangles, 32 tets
@pytest.mark.parametrize("valence", [3, 8, 9, 15, 16, 17, 24, 31, 32, 33, 47, 100])
@pytest.mark.parametrize("make,cls", [(_fan, TriaMesh), (_spindle, TetMesh)])
def test_pattern_of_high_valence(valence, make, cls):
    v, t = make(valence)
    s = Solver(cls(v, t))
    n = len(v)
    want = np.zeros((n, n), bool)
    for q in range(t.shape[1]):
        for r in range(t.shape[1]):
            want[t[:, q], t[:, r]] = True
    a = s.stiffness.tocsr()
    rows = [np.flatnonzero(want[i]) for i in range(n)]
    assert np.array_equal(a.indices, np.concatenate(rows))
    assert np.array_equal(np.diff(a.indptr), [len(r) for r in rows])


# 2 n - 3 edges: leaves of fewer than 8, of 128 and less, whole and partial
# buffers of 8192
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [3, 5, 6, 65, 66, 67, 70, 133, 1030, 4096, 4097, 4098, 4101, 8195, 40001])
def test_mean_edge_length_bits(n, dtype):
    rng = np.random.default_rng(n)
    i = np.arange(n)
    v = np.c_[0.5 * i, i % 2, np.zeros(n)] + 0.2 * rng.standard_normal((n, 3))
    v = v.astype(dtype)
    t = np.c_[i[:-2], i[1:-1], i[2:]]
    t[1::2] = t[1::2][:, [1, 0, 2]]
    assert TriaMesh(v, t).avg_edge_length() == fem.avg_edge_length(v, t)
