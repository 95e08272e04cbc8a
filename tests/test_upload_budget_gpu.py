"""An input whose columns fit the pool's budget is uploaded within it: rows on
their way take a bounded buffer, not a second copy of the input."""

import ctypes

import numpy as np
import pytest

from srdatalog_hip import native, programs

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def test_upload_within_the_columns_and_a_bounded_buffer():
  n = 30_000_001                                 # columns of 229 MiB
  rows = np.arange(2 * n, dtype=np.uint32).reshape(n, 2)
  lib = programs.load("triangle")
  set_budget = native.load_runtime()._ZN3srd15pool_set_budgetEm
  set_budget.argtypes, set_budget.restype = [ctypes.c_uint64], None
  assert lib.init() == 0
  try:
    set_budget(native.pool_stats()["in_use"] + 380 * MIB)
    lib.load_rows("KnowsInput", rows)
    assert lib.lib.srdatalog_prepare() == 0
    set_budget(0)
    assert lib.run(0) == 0
    assert np.array_equal(lib.export("Knows", 2), rows)
  finally:
    set_budget(0)
    lib.shutdown()
