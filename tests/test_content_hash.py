"""The content hash that ties a device mesh to a mesh object's arrays: equal
for equal contents, different after any single change, at sizes around its
blocks (1 KiB), segments (1 MiB) and thread counts, wherever the array starts."""

import numpy as np
import pytest

from lapy_amd import _lib
from lapy_amd.mesh import _fingerprint


@pytest.mark.parametrize("nbytes", [0, 1, 15, 16, 1023, 1024, 1025, (1 << 20) - 1, 1 << 20, (1 << 20) + 1,
                                    (6 << 20) + 517, 20 << 20])
def test_hash_sees_every_byte(nbytes):
    rng = np.random.default_rng(nbytes)
    a = rng.integers(0, 256, nbytes, dtype=np.uint8)
    h = _lib.content_hash(a)
    assert _lib.content_hash(a.copy()) == h
    shifted = np.empty(nbytes + 3, np.uint8)[3:]  # not aligned to a word
    shifted[:] = a
    assert _lib.content_hash(shifted) == h
    places = {0, nbytes // 2, nbytes - 1} | set(rng.integers(0, max(nbytes, 1), 8).tolist()) if nbytes else set()
    for p in places:
        b = a.copy()
        b[p] ^= 1 << int(rng.integers(8))
        assert _lib.content_hash(b) != h
    assert _lib.content_hash(np.append(a, np.uint8(0))) != h  # the padding's value, another size


def test_hash_sees_order():
    a = np.arange(40_000, dtype=np.uint64)
    h = _lib.content_hash(a)
    for i, j in ((0, 1), (0, 128), (5, 39_999), (1 << 14, (1 << 14) + 131_072 // 8)):  # within and across blocks, segments
        b = a.copy()
        b[[i, j]] = b[[j, i]]
        assert _lib.content_hash(b) != h


def test_fingerprint_sees_type_and_shape():
    v = np.zeros((4, 3))
    t = np.zeros((2, 3), dtype=np.int64)
    keys = {_fingerprint(v, t), _fingerprint(v.astype(np.float32), t), _fingerprint(v.reshape(3, 4), t),
            _fingerprint(v, t.astype(np.int32)), _fingerprint(v, t.reshape(3, 2)), _fingerprint(v + 0.0, t + 1)}
    assert len(keys) == 6
