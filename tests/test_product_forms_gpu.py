"""The rules of the `products` program against numpy: every form of a rule that
ends in a product, marked row by row or by unions where it may be, and with
each of these ways off."""

import numpy as np
import pytest

from srdatalog_hip import programs

pytestmark = pytest.mark.gpu

SETTINGS = {"default": {}, "tuples": {"SRDATALOG_MARK_PRODUCTS": "0"},
            "no-union": {"SRDATALOG_MARK_UNION": "0"}, "rows": {"SRDATALOG_DENSE_MAX_BITS": "0"}}


def inputs(seed, dense):
  """Few keys with products of hundreds to thousands of tuples, ids below 400
  (so that four columns are marked too)."""
  rng = np.random.default_rng(seed)
  keys, top = 9, 400

  def rel(n_left, n_right, rows):
    e = np.stack([rng.integers(0, n_left, rows), rng.integers(0, n_right, rows)], 1)
    return np.unique(e.astype(np.uint32), axis=0)

  rows = 2000 if dense else 60
  return {"A": rel(keys, top, rows), "B": rel(top, top, 4 * rows), "C": rel(keys, top, rows),
          "U": np.array([[0], [2], [3], [7]], np.uint32),
          "S": np.unique(rng.integers(0, top, 200 if dense else 9).astype(np.uint32)).reshape(-1, 1)}


def by_key(rows):
  out = {}
  for k, v in rows.tolist():
    out.setdefault(k, []).append(v)
  return out


def model(i):
  """Relation -> set of tuples."""
  a, b, c = by_key(i["A"]), by_key(i["B"]), by_key(i["C"])
  u = set(i["U"][:, 0].tolist())
  s = i["S"][:, 0].tolist()
  return {
    "Indep": {(x, y) for r in a if r in u for x in a[r] for y in s},
    "IndepKey": {(r, x, y) for r in a if r in u for x in a[r] for y in s},
    "RootNeg": {(x, y) for r in a if r in c and r not in u for x in a[r] for y in c[r]},
    "RootFilter": {(x, y) for r in a if r in c and r != 3 for x in a[r] for y in c[r]},
    "RootTwice": {(r, r, x, y) for r in a if r in c
                  for x in {v for m in a[r] for v in b.get(m, ())} for y in c[r]},
    "KeyUnion": {(r, x, y) for r in a if r in c
                 for x in {v for m in a[r] for v in b.get(m, ())} for y in c[r]},
    "KeyUnionMinor": {(y, r, x) for r in a if r in c
                      for x in {v for m in a[r] for v in b.get(m, ())} for y in c[r]},
    "Deep": {(x, y) for r in a if r in c
             for x in {v for m in a[r] for z in b.get(m, ()) for v in b.get(z, ())} for y in c[r]},
  }


@pytest.mark.parametrize("setting", SETTINGS)
@pytest.mark.parametrize("seed,dense", [(0, True), (1, True), (2, False)])
def test_product_forms_match_numpy(seed, dense, setting, monkeypatch):
  for k, v in SETTINGS[setting].items():
    monkeypatch.setenv(k, v)
  i = inputs(seed, dense)
  lib = programs.load("products")
  assert lib.init() == 0
  try:
    for name, rows in i.items():
      lib.load_rows(name, rows)
    assert lib.run(0) == 0
    for rel, want in model(i).items():
      k = len(next(iter(want)))
      got = lib.export(rel, k)
      assert np.array_equal(got, np.array(sorted(want), np.uint32).reshape(-1, k)), rel
  finally:
    lib.shutdown()
