"""The one-launch sort of small inputs (small_sort_kernel) at the edges of its
waves, items and key words, against numpy: rows, root arrays, repeats, equal
digits, single values; the row counts around its limit take both paths."""

import numpy as np
import pytest

from srdatalog_hip import native

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 1000, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 5000]


@pytest.mark.parametrize("k", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["wide", "narrow", "high-only", "equal", "sorted"])
def test_small_sorts(kind, k):
  rng = np.random.default_rng(k)
  for n in SIZES:
    if kind == "wide":
      rows = rng.integers(0, 2**32, size=(n, k), dtype=np.uint64).astype(np.uint32)
      rows[n // 2:] = rows[rng.integers(0, n, size=n - n // 2)]
    elif kind == "narrow":
      rows = rng.integers(0, 9, size=(n, k), dtype=np.uint64).astype(np.uint32)
    elif kind == "high-only":
      rows = (rng.integers(0, 200, size=(n, k), dtype=np.uint64) << np.uint64(24)).astype(np.uint32)
    elif kind == "equal":
      rows = np.full((n, k), 0xFFFFFFFF, np.uint32)
    else:
      rows = np.unique(rng.integers(0, 2**20, size=(n, k), dtype=np.uint64).astype(np.uint32), axis=0)
    want = np.unique(rows, axis=0)
    got, vals, offs = native.sort_dedup(rows)
    assert np.array_equal(got, want), n
    v, first = np.unique(want[:, 0], return_index=True)
    assert np.array_equal(vals, v) and np.array_equal(offs, np.append(first, want.shape[0])), n
