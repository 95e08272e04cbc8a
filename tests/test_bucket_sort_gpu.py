"""The two-launch sort of 4,097 to 2^20 rows (bucket_part_kernel,
bucket_sort_kernel) against numpy: row counts at the edges of its bucket and
tile rules, key widths, values that repeat across splitters, and rows chosen
so that the sample misses them, which leaves one bucket far beyond LDS."""

import numpy as np
import pytest

from srdatalog_hip import native

pytestmark = pytest.mark.gpu

SIZES = [4097, 8191, 8192, 16385, 99_991, 262_143, 262_145, 524_289, (1 << 20) - 1, 1 << 20]


def check(rows):
  n = rows.shape[0]
  want = np.unique(rows, axis=0)
  got, vals, offs = native.sort_dedup(rows)
  assert np.array_equal(got, want), n
  v, first = np.unique(want[:, 0], return_index=True)
  assert np.array_equal(vals, v) and np.array_equal(offs, np.append(first, want.shape[0])), n


def values(rng, kind, n, k):
  if kind == "wide":
    return rng.integers(0, 2**32, size=(n, k), dtype=np.uint64).astype(np.uint32)
  if kind == "narrow":   # every value many times over
    return rng.integers(0, max(2, int(3000 ** (1 / k))), size=(n, k), dtype=np.uint64).astype(np.uint32)
  if kind == "skew":     # half the rows equal, the rest under few first values
    rows = rng.integers(0, 2**20, size=(n, k), dtype=np.uint64).astype(np.uint32)
    rows[:, 0] >>= 15
    rows[rng.random(n) < 0.5] = 0xFFFFFFFF
    return rows
  return np.unique(rng.integers(0, 2**32, size=(n, k), dtype=np.uint64).astype(np.uint32), axis=0)


@pytest.mark.parametrize("k", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["wide", "narrow", "skew", "sorted"])
def test_bucket_sorts(kind, k):
  rng = np.random.default_rng(k)
  for n in SIZES:
    print(kind, k, n, flush=True)
    check(values(rng, kind, n, k))


def sampled(n):
  """Rows that bucket_part_kernel samples."""
  bins = 8
  while bins < 512 and bins * 1024 <= n:
    bins *= 2
  s = max(8 * bins, 1024)
  j = np.arange(s, dtype=np.uint64)
  step = np.uint64((n << 11) // s)
  h = (j * np.uint64(2654435761) & np.uint64(0xFFFFFFFF)) >> np.uint64(16)
  return ((j * step >> np.uint64(11)) + (h * (step >> np.uint64(11)) >> np.uint64(16))).astype(np.int64)


@pytest.mark.parametrize("k", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [20_000, 100_003])
def test_bucket_beyond_lds(n, k):
  rng = np.random.default_rng(n + k)
  # what the sample sees is below 2^16, everything else above it
  rows = rng.integers(1 << 16, 1 << 20, size=(n, k), dtype=np.uint64).astype(np.uint32)
  rows[:n // 8] = rows[rng.integers(0, n, size=n // 8)]
  at = sampled(n)
  rows[at] = rng.integers(0, 1 << 16, size=(at.size, k), dtype=np.uint64).astype(np.uint32)
  check(rows)
