"""Rules that copy a relation share the index they read (pr_copy): relations,
deltas and derivation counts against the oracle and against the same run with
every row derived, over inputs with repeats, without rows and in order, run
twice in one session."""

import numpy as np
import pytest

import oracle
from srdatalog_hip import programs

pytestmark = pytest.mark.gpu


def run(prog, inputs, rel, k, times=1):
  lib = programs.load(prog)
  assert lib.init() == 0
  try:
    for name, rows in inputs.items():
      lib.load_rows(name, rows)
    for _ in range(times):
      assert lib.run(0) == 0
    return lib.export(rel, k), lib.delta_sizes(rel), lib.join_tuples()
  finally:
    lib.shutdown()


def edges(kind):
  rng = np.random.default_rng(3)
  if kind == "none":
    return np.empty((0, 2), np.uint32)
  if kind == "one":
    return np.array([[7, 9]], np.uint32)
  rows = rng.integers(0, 300, size=(6000, 2), dtype=np.uint64).astype(np.uint32)
  if kind == "sorted":
    return np.unique(rows, axis=0)
  return np.concatenate([rows, rows[::3]])


@pytest.mark.parametrize("kind", ["none", "one", "sorted", "repeats"])
@pytest.mark.parametrize("prog,inp,rel,k", [("triangle", "KnowsInput", "Triangle", 3),
                                            ("tc", "ArcInput", "Path", 2)])
def test_copies_match_derived_rows(prog, inp, rel, k, kind, monkeypatch):
  rows = edges(kind)
  shared = run(prog, {inp: rows}, rel, k, times=2)
  monkeypatch.setenv("SRDATALOG_COPY_SHARE", "0")
  derived = run(prog, {inp: rows}, rel, k, times=2)
  want = oracle.run(prog, {inp: rows})
  assert np.array_equal(shared[0], want.relations[rel]) and np.array_equal(derived[0], shared[0])
  assert shared[1] == derived[1] and shared[2] == derived[2]
