"""Inputs that are split into columns on the device: sizes around the limit
and around the copied pieces, arities, unaligned row pointers, replaced
inputs, rows changed by the caller after the load, and CSV files."""

import ctypes

import numpy as np
import pytest

import oracle
from srdatalog_hip import programs

pytestmark = pytest.mark.gpu

LIMIT = 1 << 16   # rows of two columns that go to the device at once


def session(rows, offset=0):
  lib = programs.load("triangle")
  assert lib.init() == 0
  try:
    lib.load_rows("KnowsInput", np.array([[0, 1]], np.uint32))   # replaced below
    words = np.empty(rows.size + offset, np.uint32)[offset:]
    words[:] = rows.reshape(-1)
    p = words.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))
    assert lib.lib.srdatalog_load_rows(b"KnowsInput", p, rows.shape[0], 2) == 0
    assert lib.size("KnowsInput") == rows.shape[0]
    words[:] = 0   # the load has consumed them
    assert lib.run(0) == 0
    return lib.export("Knows", 2)
  finally:
    lib.shutdown()


@pytest.mark.parametrize("n", [LIMIT - 1, LIMIT, LIMIT + 1, (1 << 19) - 1, (1 << 19) + 1, 3_000_001])
@pytest.mark.parametrize("offset", [0, 1])
def test_pairs_reach_the_index(n, offset):
  rng = np.random.default_rng(n)
  # few edges per vertex, so that the program's join stays small
  rows = rng.integers(0, 2**31, size=(n, 2), dtype=np.uint64).astype(np.uint32)
  want = np.unique(rows, axis=0)
  assert np.array_equal(session(rows, offset), want)


def test_large_csv_and_triples(tmp_path):
  rng = np.random.default_rng(3)
  n = 70_000
  r = rng.integers(0, 300, size=(n, 3), dtype=np.uint64).astype(np.uint32)
  np.savetxt(tmp_path / "R.csv", r, fmt="%d", delimiter="\t")
  lib = programs.load("galen")
  assert lib.init() == 0
  try:
    for rel, k in (("PInput", 2), ("UInput", 3), ("CInput", 3), ("SInput", 2), ("RInput", 3)):
      lib.load_rows(rel, np.zeros((0, k), np.uint32))
    assert lib.load_csv("QInput", str(tmp_path / "R.csv")) == 0
    assert lib.run(0) == 0
    assert np.array_equal(lib.export("OutQ", 3), np.unique(r, axis=0))
  finally:
    lib.shutdown()
