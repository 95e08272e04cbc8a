"""Iterations on bitmaps (run_step_dense): relation and per-iteration deltas
against the oracle for closures, same generation and reachability, from key
spaces of a few words to several blocks, DELTA buffers that must grow, capped
iterations, packed instances, and the hand-over to the host loop."""

import numpy as np
import pytest

import oracle
from srdatalog_hip import batch, datasets, programs

pytestmark = pytest.mark.gpu

SETTINGS = {"default": {}, "grow": {"SRDATALOG_DENSE_DELTA_ROWS": "70"},
            "grain": {"SRDATALOG_GRAIN": "64"}, "tuples": {"SRDATALOG_MARK_PRODUCTS": "0"},
            "host-after-500": {"SRDATALOG_DENSE_DELTA_ROWS": "70", "SRDATALOG_DEVLOOP_MAX_ROWS": "500"}}


def run(prog, inputs, rel, arity, max_iters=0):
  lib = programs.load(prog)
  assert lib.init() == 0
  try:
    for name, rows in inputs.items():
      lib.load_rows(name, rows)
    for _ in range(2):   # the second run finds the bitmaps of the first
      assert lib.run(max_iters) == 0
      got = lib.export(rel, arity), lib.delta_sizes(rel)
    return got
  finally:
    lib.shutdown()


def cases():
  rng = np.random.default_rng(5)
  for n, m, stride in ((2, 2, 1), (40, 60, 1), (64, 200, 1), (65, 300, 1), (300, 900, 1), (300, 400, 37),
                       (500, 2500, 1), (60, 200, 1000)):
    e = datasets.tc_edges(n, n, m) * np.uint32(stride)
    yield f"tc-{n}-{m}-{stride}", "tc", {"ArcInput": e}, "Path", 2
  yield "tc-chain", "tc", {"ArcInput": np.array([[i, i + 1] for i in range(130)], np.uint32)}, "Path", 2
  yield "tc-empty", "tc", {"ArcInput": np.zeros((0, 2), np.uint32)}, "Path", 2
  for n in (30, 400, 1500):
    yield f"sg-{n}", "sg", {"Arc": datasets.sg_forest_edges(rng, n)}, "Sg", 2
  for n, m, top in ((50, 150, 0), (3000, 9000, 0), (900, 4000, 300_000)):
    e = datasets.tc_edges(n, n, m) + np.uint32(top)
    yield f"reach-{n}-{top}", "reach", {"Src": e[:1, :1].copy(), "Edge": e}, "Reach", 1


CASES = list(cases())


@pytest.mark.parametrize("setting", SETTINGS)
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_dense_iterations_match_the_oracle(case, setting, monkeypatch):
  for k, v in SETTINGS[setting].items():
    monkeypatch.setenv(k, v)
  _, prog, inputs, rel, arity = case
  want = oracle.run(prog, inputs)
  got, deltas = run(prog, inputs, rel, arity)
  assert np.array_equal(got, want.relations[rel])
  assert deltas == want.deltas[rel]


@pytest.mark.parametrize("iters", [1, 2, 5])
def test_capped_iterations(iters, monkeypatch):
  e = datasets.tc_edges(3, 200, 500)
  got = run("tc", {"ArcInput": e}, "Path", 2, iters)
  monkeypatch.setenv("SRDATALOG_DEVLOOP", "0")
  want = run("tc", {"ArcInput": e}, "Path", 2, iters)
  assert np.array_equal(got[0], want[0]) and got[1] == want[1]


def test_many_iterations_grow_the_record():
  n = 1200   # 1,200 iterations: more than the first record holds
  e = np.array([[i, i + 1] for i in range(n)], np.uint32)
  rows, deltas = run("tc", {"ArcInput": e}, "Path", 2)
  assert deltas == [n - i for i in range(1, n)] + [0]
  assert rows.shape[0] == n * (n + 1) // 2


@pytest.mark.parametrize("kind", ["tc", "sg"])
def test_packed_instances(kind):
  rng = np.random.default_rng(8)
  insts = []
  for i, n in enumerate((2, 17, 64, 65, 300, 700)):
    e = datasets.tc_edges(i, n, 2 * n if n > 2 else 1) if kind == "tc" else datasets.sg_forest_edges(rng, n)
    insts.append(batch.Instance(kind, n, e))
  for got, want in zip(batch.run_batched(kind, insts), batch.run_plain(kind, insts)):
    assert np.array_equal(got.rows, want.rows) and got.deltas == want.deltas
