"""The host side of the iterations on bitmaps (run_step_dense) against a
simulated device (tests/cpu_sim/dense_cpu.cpp): relation and deltas against
the oracle where a DELTA buffer grows while the host is still reading the
report before it."""

import ctypes

import numpy as np
import pytest

import oracle
from conftest import build_cpu_sim
from srdatalog_hip import codegen, compiler, programs
from srdatalog_hip import datasets as ds

_u32p = ctypes.POINTER(ctypes.c_uint32)


@pytest.fixture(scope="module")
def lib():
  lib = ctypes.CDLL(build_cpu_sim("libdense_cpu.so"))
  for f in ("cpu_dense_engine", "cpu_union_engine"):
    getattr(lib, f).restype = ctypes.c_void_p
    getattr(lib, f).argtypes = [ctypes.c_char_p]
  lib.srd_engine_ok.argtypes = [ctypes.c_void_p]
  lib.srd_engine_load_rows.argtypes = [ctypes.c_void_p, ctypes.c_char_p, _u32p, ctypes.c_uint64,
                                       ctypes.c_uint32]
  lib.srd_engine_run.argtypes = [ctypes.c_void_p, ctypes.c_ulonglong]
  lib.srd_engine_export.argtypes = [ctypes.c_void_p, ctypes.c_char_p, _u32p, ctypes.c_uint64,
                                    ctypes.POINTER(ctypes.c_uint64)]
  lib.srd_engine_delta_sizes.argtypes = [ctypes.c_void_p, ctypes.c_char_p,
                                         ctypes.POINTER(ctypes.c_ulonglong), ctypes.c_ulonglong]
  lib.srd_engine_destroy.argtypes = [ctypes.c_void_p]
  lib.srd_engine_set_quiet.argtypes = [ctypes.c_void_p, ctypes.c_int]
  lib.sim_fail_alloc.argtypes = [ctypes.c_uint64, ctypes.c_uint64]
  for f in ("sim_split_report", "sim_fail_book", "sim_pool_limit"):
    getattr(lib, f).argtypes = [ctypes.c_uint64]
  for f in ("sim_pool_used", "sim_late_writes", "sim_dense_iterations", "sim_size_after_failure",
            "sim_allocs_to_failure"):
    getattr(lib, f).restype = ctypes.c_uint64
  return lib


@pytest.fixture(autouse=True)
def plain_settings(monkeypatch, lib):
  for k in ("DEVLOOP", "DEVLOOP_GRAPH", "DEVLOOP_CAPS", "DEVLOOP_BATCH", "DEVLOOP_MAX_BYTES",
            "DEVLOOP_MAX_ROWS", "DEVLOOP_DENSE", "DENSE_DELTA_ROWS", "DENSE_MAX_BITS", "JOIN_MODE"):
    monkeypatch.delenv("SRDATALOG_" + k, raising=False)
  lib.sim_reset()


class Engine:
  def __init__(self, lib, make):
    prog = programs.tc_program()
    text = codegen.program_text(compiler.relation_decls(prog), compiler.compile_to_mir(prog))
    self.lib, self.e = lib, ctypes.c_void_p(make(text.encode()))
    assert lib.srd_engine_ok(self.e) == 1
    lib.srd_engine_set_quiet(self.e, 1)

  def run(self, edges, max_iters=0):
    edges = np.ascontiguousarray(edges, dtype=np.uint32)
    self.lib.srd_engine_load_rows(self.e, b"ArcInput", edges.ctypes.data_as(_u32p), edges.shape[0], 2)
    return self.lib.srd_engine_run(self.e, max_iters)

  def path(self):
    n = ctypes.c_uint64()
    self.lib.srd_engine_export(self.e, b"Path", None, 0, ctypes.byref(n))
    out = np.empty((max(n.value, 1), 2), np.uint32)
    self.lib.srd_engine_export(self.e, b"Path", out.ctypes.data_as(_u32p), n.value, ctypes.byref(n))
    cnt = self.lib.srd_engine_delta_sizes(self.e, b"Path", None, 0)
    buf = (ctypes.c_ulonglong * max(cnt, 1))()
    self.lib.srd_engine_delta_sizes(self.e, b"Path", buf, cnt)
    return out[:n.value], [int(buf[i]) for i in range(cnt)]

  def close(self):
    self.lib.srd_engine_destroy(self.e)


@pytest.fixture
def engine(lib):
  engines = []

  def make(kind=lib.cpu_dense_engine):
    engines.append(Engine(lib, kind))
    return engines[-1]
  yield make
  for e in engines:
    e.close()


def check(got, edges, max_iters=0):
  want = oracle.run("tc", {"ArcInput": edges}, **({"max_iters": max_iters} if max_iters else {}))
  np.testing.assert_array_equal(got[0], want.relations["Path"])
  assert got[1] == want.deltas["Path"]


def fan(width, tail):
  """`width` sources into a chain of two, out to `width` targets that all
  enter a chain of `tail`: the first iteration derives few pairs, the second
  width * width of them."""
  s, t = np.arange(width), 100 + np.arange(width)
  chain = [(50, 51)] + [(200 + i, 201 + i) for i in range(tail)]
  return np.array([(a, 50) for a in s] + [(51, b) for b in t] + [(b, 200) for b in t] + chain, np.uint32)


@pytest.mark.parametrize("n,m,seed", [(2, 2, 0), (40, 60, 1), (200, 500, 2), (600, 1500, 3)])
def test_bitmap_iterations_match_the_oracle(lib, engine, n, m, seed):
  e = ds.tc_edges(seed, n, m)
  eng = engine()
  for _ in range(2):
    assert eng.run(e) == 0
    check(eng.path(), e)
  assert eng.run(e, 2) == 0
  check(eng.path(), e, 2)
  assert lib.sim_dense_iterations() > 0 and lib.sim_late_writes() == 0


def test_growing_delta_while_the_report_is_half_there(lib, engine, monkeypatch):
  """The second iteration overflows DELTA; the host takes the first one's
  report while the second's flag is already stored and its count is not."""
  monkeypatch.setenv("SRDATALOG_DENSE_DELTA_ROWS", "128")
  e = fan(30, 20)
  lib.sim_split_report(2)
  eng = engine()
  assert eng.run(e) == 0
  check(eng.path(), e)


def test_a_buffer_that_could_not_grow_is_empty(lib):
  """Not a size without memory, which the next reserve would take for a
  buffer of that size."""
  assert lib.sim_size_after_failure() == 0


@pytest.mark.parametrize("nth", [1, 2, 4])
def test_a_run_after_a_failed_one_starts_clear(lib, engine, nth):
  """A launch fails in the middle of the iterations: the marks that the failed
  run left in NEW are no part of the next one."""
  eng = engine()
  lib.sim_fail_book(nth)
  assert eng.run(ds.tc_edges(4, 50, 200)) != 0
  lib.sim_fail_book(0)
  e = ds.tc_edges(5, 40, 60)
  assert eng.run(e) == 0
  check(eng.path(), e)


def test_a_failed_run_keeps_its_pinned_block_until_the_launches_ran(lib, engine):
  """The third iteration cannot be launched; the first two are still to run
  and report into the block."""
  eng = engine()
  lib.sim_hold()
  lib.sim_fail_book(3)
  assert eng.run(ds.tc_edges(4, 50, 200)) != 0
  lib.sim_fail_book(0)
  e = ds.tc_edges(5, 40, 60)
  assert eng.run(e) == 0
  check(eng.path(), e)
  assert lib.sim_late_writes() == 0


def test_no_iterations_on_bitmaps_above_the_memory_budget(lib, engine, monkeypatch):
  monkeypatch.setenv("SRDATALOG_DEVLOOP_MAX_BYTES", str(1 << 20))
  e = ds.tc_edges(6, 500, 900)
  eng = engine()
  assert eng.run(e) == 0
  check(eng.path(), e)
  assert lib.sim_dense_iterations() == 0


def test_no_iterations_on_bitmaps_without_memory_for_them(lib, engine):
  """The pool holds the relations but not the DELTA buffer of 2^20 keys."""
  e = ds.tc_edges(6, 1000, 1500)
  eng = engine()
  lib.sim_pool_limit(lib.sim_pool_used() + (8 << 20))
  assert eng.run(e) == 0
  check(eng.path(), e)
  assert lib.sim_dense_iterations() == 0
  lib.sim_pool_limit(0)
  assert eng.run(e) == 0
  check(eng.path(), e)
  assert lib.sim_dense_iterations() > 0


def test_growth_above_the_memory_budget_hands_over(lib, engine, monkeypatch):
  """DELTA of 90,000 rows and more does not fit a megabyte: the second
  iteration and those after it run on the host loop."""
  monkeypatch.setenv("SRDATALOG_DENSE_DELTA_ROWS", "1300")
  monkeypatch.setenv("SRDATALOG_DEVLOOP_MAX_BYTES", str(1 << 20))
  w, tail = 300, 12
  s, t = np.arange(w), 300 + np.arange(w)
  e = np.concatenate([np.stack([s, np.full(w, 900)], 1), [[900, 901]], np.stack([np.full(w, 901), t], 1),
                      np.stack([t, np.full(w, 910)], 1),
                      np.stack([910 + np.arange(tail), 911 + np.arange(tail)], 1)]).astype(np.uint32)
  eng = engine()
  assert eng.run(e) == 0
  check(eng.path(), e)
  assert 2 <= lib.sim_dense_iterations() <= 4    # what was sent ahead of the overflow


@pytest.mark.parametrize("nth", [1, 2, 3])
def test_growth_without_memory_hands_over(lib, engine, monkeypatch, nth):
  """One buffer of the larger DELTA (columns, root values, root offsets) cannot
  be had: the last whole DELTA goes to the host loop."""
  monkeypatch.setenv("SRDATALOG_DENSE_DELTA_ROWS", "128")
  e = fan(30, 20)
  eng = engine()
  lib.sim_fail_alloc(nth, 0)
  assert eng.run(e) == 0
  assert lib.sim_allocs_to_failure() == 0
  check(eng.path(), e)
  assert lib.sim_dense_iterations() <= 4
  assert eng.run(e) == 0                          # and with the memory back
  check(eng.path(), e)


def test_a_union_without_memory_leaves_the_rule_to_mark(lib, engine, monkeypatch):
  """Ids below 1,024: NEW's bitmap and the unions' are 128 KiB each, and the
  second of them cannot be had in any iteration."""
  monkeypatch.setenv("SRDATALOG_DEVLOOP", "0")
  e = ds.tc_edges(7, 600, 900)
  eng = engine(lib.cpu_union_engine)
  lib.sim_fail_alloc(2, 1 << 17)
  # one iteration: the next would find the memory
  assert eng.run(e, 1) == 0
  assert lib.sim_allocs_to_failure() == 0
  check(eng.path(), e, 1)


def test_rows_that_cannot_be_loaded_leave_the_ones_there(lib, engine):
  """A load that neither the device nor the host has memory for."""
  e = ds.tc_edges(8, 60, 100)
  eng = engine()
  assert eng.run(e) == 0
  lib.sim_pool_limit(lib.sim_pool_used() + (1 << 20))
  assert lib.srd_engine_load_rows(eng.e, b"ArcInput", e.ctypes.data_as(_u32p), 1 << 60, 2) != 0
  lib.sim_pool_limit(0)
  assert lib.srd_engine_run(eng.e, 0) == 0
  check(eng.path(), e)


def test_rows_the_device_cannot_split_are_split_on_the_host(lib, engine, monkeypatch):
  """Neither at the load nor at the run is there pinned memory for rows on
  their way to the device; the columns need none."""
  monkeypatch.setenv("SRDATALOG_DEVLOOP", "0")
  n = 1 << 16                                     # pairs: the smallest input sent as rows
  e = np.stack([np.arange(n), n + np.arange(n)], 1).astype(np.uint32)
  eng = engine()
  lib.sim_set_upload_fails(1)
  assert eng.run(e) == 0
  got = eng.path()
  np.testing.assert_array_equal(got[0], e)
  assert got[1] == [0]
