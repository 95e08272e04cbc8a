"""Iterations on bitmaps within SRDATALOG_DEVLOOP_MAX_BYTES: no bitmaps above
it, and a DELTA that may not grow hands the step to the host loop; relation
and deltas against the oracle either way."""

import numpy as np
import pytest

import oracle
from srdatalog_hip import datasets, programs

pytestmark = pytest.mark.gpu


# 700 vertices: the bitmaps of 2^20 keys, the key buffers and the first DELTA
# are 0.32 MB, above the first limit; the fourth iteration's 48,384 rows of
# DELTA are above the second; the third holds everything
@pytest.mark.parametrize("limit", [100_000, 1_000_000, 1 << 26])
def test_closure_within_a_memory_budget(limit, monkeypatch):
  monkeypatch.setenv("SRDATALOG_DEVLOOP_MAX_BYTES", str(limit))
  monkeypatch.setenv("SRDATALOG_DENSE_DELTA_ROWS", "2000")
  e = datasets.tc_edges(9, 700, 1750)
  want = oracle.run("tc", {"ArcInput": e})
  lib = programs.load("tc")
  assert lib.init() == 0
  try:
    lib.load_rows("ArcInput", e)
    for _ in range(2):   # the second run finds what the first left
      assert lib.run(0) == 0
      assert np.array_equal(lib.export("Path", 2), want.relations["Path"])
      assert lib.delta_sizes("Path") == want.deltas["Path"]
  finally:
    lib.shutdown()
