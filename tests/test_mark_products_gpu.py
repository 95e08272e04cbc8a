"""Products marked row by row (srdj::prod_mark) at the edges of its pairs and
rows: 64 pairs to a flush, 64 rows to a step, dense and sparse last columns,
products split between slices; relation and deltas against the oracle, and
the same with the products marked tuple by tuple or per level-1 value
instead of once per root key over the union of its values."""

import numpy as np
import pytest

import oracle
from srdatalog_hip import datasets, programs

pytestmark = pytest.mark.gpu

SETTINGS = [{}, {"SRDATALOG_MARK_PRODUCTS": "0"}, {"SRDATALOG_MARK_UNION": "0"},
            {"SRDATALOG_MARK_UNION": "0", "SRDATALOG_GRAIN": "65"},
            {"SRDATALOG_WEIGH_TARGET": "1024", "SRDATALOG_MIN_SLICES_PER_WAVE": "1"}]
SHAPES = [(1, 300), (300, 1), (63, 64), (64, 65), (65, 128), (129, 127), (400, 700)]


def run(prog, inputs, rel):
  lib = programs.load(prog)
  assert lib.init() == 0
  try:
    for name, rows in inputs.items():
      lib.load_rows(name, rows)
    assert lib.run(0) == 0
    return lib.export(rel, 2), lib.delta_sizes(rel)
  finally:
    lib.shutdown()


def pairs(a, b):
  return np.array([(x, y) for x in a for y in b], dtype=np.uint32).reshape(-1, 2)


@pytest.mark.parametrize("env", SETTINGS, ids=["default", "tuples", "no-union", "grain-65", "small-slices"])
@pytest.mark.parametrize("stride", [1, 3, 70])
def test_products_match_the_oracle(stride, env, monkeypatch):
  monkeypatch.setenv("SRDATALOG_DEVLOOP", "0")   # the host loop marks
  for k, v in env.items():
    monkeypatch.setenv(k, v)
  for a, b in SHAPES:
    # a sources and b targets around one hub, a second hop behind the targets
    src = 5 + stride * np.arange(a)
    dst = 5 + stride * (a + np.arange(b)) + 1
    hub = int(dst[-1]) + 7
    edges = np.concatenate([pairs(src, [hub]), pairs([hub], dst), pairs(dst[:3], [hub + 1])])
    want = oracle.run("tc", {"ArcInput": edges})
    got, deltas = run("tc", {"ArcInput": edges}, "Path")
    assert np.array_equal(got, want.relations["Path"]) and deltas == want.deltas["Path"], (a, b)
    # *x = y and y = *x: every target of x takes every object of y
    x, y = hub + 2, hub + 3
    z = hub + 4
    inputs = {"AddressOf": np.concatenate([pairs([x], src), pairs([y], dst)]),
              "Assign": pairs([z], [x]), "Load": pairs([z, z + 1], [x]), "Store": pairs([x], [y])}
    want = oracle.run("andersen", inputs)
    got, deltas = run("andersen", inputs, "PointsTo")
    assert np.array_equal(got, want.relations["PointsTo"]) and deltas == want.deltas["PointsTo"], (a, b)


@pytest.mark.parametrize("env", SETTINGS[:3], ids=["default", "tuples", "no-union"])
@pytest.mark.parametrize("seed,div", [(0, 700), (1, 300), (2, 90)])
def test_unions_match_the_oracle(seed, div, env, monkeypatch):
  """Zipf points-to: root keys with one and with thousands of level-1 values."""
  for k, v in env.items():
    monkeypatch.setenv(k, v)
  inputs = datasets.andersen_inputs(seed, 200_000 // div, 50_000 // div,
                                    (100_000 // div, 400_000 // div, 100_000 // div, 100_000 // div))
  want = oracle.run("andersen", inputs)
  got, deltas = run("andersen", inputs, "PointsTo")
  assert np.array_equal(got, want.relations["PointsTo"]) and deltas == want.deltas["PointsTo"]
