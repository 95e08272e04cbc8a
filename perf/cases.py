"""The work whose time is tracked: calls of the framework's public entry points.

Two kinds of call.  ``sort`` is the set primitive on device columns
(``srd_prim_sort_dedup_noalloc``), the one entry point that takes and returns
device buffers.  Every other case is a whole session of a compiled program
as ``srdatalog_hip.runtime`` drives it -- init, load rows from host arrays,
run to the fixpoint, export the result and its per-iteration delta sizes,
shutdown -- on one input or on a packed batch of them.  A program library
holds one session at a time, so a session takes host arrays and fills the
caller's host arrays.

All results are whole numbers and compared exactly.
"""

import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "srdatalog-python_amd"))
os.environ.setdefault("SRDATALOG_QUIET", "1")   # no size lines on stdout

from srdatalog_hip import batch, datasets, native, programs  # noqa: E402


def listed():
  return [
    # The index build alone.  A small serving request's rows: launches and
    # latency, no bandwidth.
    {"name": "sort_1k", "path": "sort", "n": 1000, "k": 2, "bits": 16},
    # Triples of a mid-sized relation (two-word keys, a ragged row count).
    {"name": "sort_100k_k3", "path": "sort", "n": 99_991, "k": 3, "bits": 24},
    # The largest input the entry point takes, pairs over 2^20 ids.
    {"name": "sort_1m", "path": "sort", "n": 1 << 20, "k": 2, "bits": 20},
    # A small closure: the size of the smoke run, session overheads count.
    {"name": "tc_small", "path": "tc", "n": 400, "m": 1200},
    # Transitive closure at the benchmark's size (5,000 pairs, 1,000 vertices).
    {"name": "tc_c1", "path": "tc", "n": 1000, "m": 5000},
    # Same generation over a random forest, an instance of the uneven batch.
    {"name": "sg_6k", "path": "sg", "n": 6000},
    # An uneven batch of closures packed into one fixpoint.
    {"name": "tc_batch_32", "path": "tc_batch", "count": 32, "n_lo": 200, "n_hi": 1500},
    # Andersen points-to at two scales: four mutually recursive rules, far
    # more derivations than tuples.
    {"name": "andersen_30", "path": "andersen", "div": 30},
    {"name": "andersen_10", "path": "andersen", "div": 10},
    # Triangle listing on an R-MAT graph (a request of the serving mix).
    {"name": "tri_list_14", "path": "triangle", "scale": 14, "factor": 16},
    # Triangle count on the benchmark's graph: R-MAT scale 20, 2^24 draws.
    {"name": "tri_count_20", "path": "triangle_count", "scale": 20, "factor": 16},
    # Single-source reachability on a base graph of the serving mix.
    {"name": "reach_18", "path": "reach", "scale": 18, "factor": 16},
  ]


def _log_int(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  path = rng.choice(["sort", "sort", "tc", "tc", "sg", "tc_batch", "andersen", "triangle",
                     "triangle_count", "reach"])
  if path == "sort":
    return {"path": path, "n": _log_int(rng, 1000, 1 << 20), "k": rng.randint(1, 4),
            "bits": rng.randint(10, 32)}
  if path == "tc":
    n = _log_int(rng, 200, 1500)
    return {"path": path, "n": n, "m": int(n * rng.uniform(1.5, 5.0))}
  if path == "sg":
    return {"path": path, "n": _log_int(rng, 500, 7000)}
  if path == "tc_batch":
    lo = _log_int(rng, 100, 500)
    return {"path": path, "count": rng.randint(8, 40), "n_lo": lo, "n_hi": 3 * lo}
  if path == "andersen":
    return {"path": path, "div": _log_int(rng, 10, 300)}
  return {"path": path, "scale": rng.randint(11, {"triangle": 15, "triangle_count": 19, "reach": 19}[path]),
          "factor": rng.randint(4, 16)}


# ------------------------------------------------------------------ inputs ----
def _rmat(scale, factor, seed, oriented):
  """Distinct loop-free R-MAT pairs (a, b, c, d) = (0.57, 0.19, 0.19, 0.05),
  drawn on the GPU; oriented low->high when asked; rows in random order."""
  g = torch.Generator(device="cuda").manual_seed(seed)
  n = factor << scale
  u = torch.zeros(n, dtype=torch.int64, device="cuda")
  v = torch.zeros_like(u)
  for _ in range(scale):
    r = torch.rand(n, generator=g, device="cuda")
    u = 2 * u + (r >= 0.76)
    v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
  keep = u != v
  u, v = u[keep], v[keep]
  if oriented:
    u, v = torch.minimum(u, v), torch.maximum(u, v)
  keys = torch.unique((u << 32) | v)
  keys = keys[torch.randperm(keys.numel(), generator=g, device="cuda")]
  rows = torch.stack([keys >> 32, keys & 0xFFFFFFFF], dim=1).to(torch.int32)
  return rows.cpu().numpy().view(np.uint32)


def _batch_instances(case, seed):
  rng = np.random.default_rng(seed)
  out = []
  for _ in range(case["count"]):
    n = int(round(math.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
    m = int(round(n * rng.uniform(1.5, 4.0)))
    out.append(batch.Instance("tc", n, datasets.tc_edges(int(rng.integers(1 << 62)), n, m)))
  return out


def _sort_columns(case, seed):
  n, k, bits = case["n"], case["k"], case["bits"]
  g = torch.Generator(device="cuda").manual_seed(seed)
  cols = torch.randint(0, 1 << bits, (k, n), generator=g, device="cuda", dtype=torch.int64)
  # one row in eight repeats another, as derivations of a join do
  dup = torch.randint(0, n, (n // 8,), generator=g, device="cuda")
  cols[:, :n // 8] = cols[:, dup]
  return torch.where(cols >= 1 << 31, cols - (1 << 32), cols).to(torch.int32)


# path -> (program, its input relation, result relation, arity of the result)
_SESSIONS = {"tc": ("tc", "ArcInput", "Path", 2), "sg": ("sg", "Arc", "Sg", 2),
             "tc_batch": ("tc", "ArcInput", "Path", 2),
             "andersen": ("andersen", None, "PointsTo", 2),
             "triangle": ("triangle", "KnowsInput", "Triangle", 3),
             "triangle_count": ("triangle_count", "KnowsInput", "Triangle", 0),
             "reach": ("reach", "Edge", "Reach", 1)}
_ITERS = 256   # rows kept for the per-iteration delta sizes


def prepare(case, seed):
  path = case["path"]
  if path == "sort":
    n, k = case["n"], case["k"]
    cols = _sort_columns(case, seed)
    return {"path": path, "lib": native.load_runtime(), "n": n, "k": k, "cols": cols,
            "out": torch.zeros_like(cols),
            "root_vals": torch.zeros(n, dtype=torch.int32, device="cuda"),
            "root_offs": torch.zeros(n + 1, dtype=torch.int32, device="cuda"),
            "counts": torch.zeros(3, dtype=torch.int64, device="cuda")}
  program, rel_in, rel_out, arity = _SESSIONS[path]
  bounds = None
  if path == "tc":
    inputs = {rel_in: datasets.tc_edges(seed, case["n"], case["m"])}
  elif path == "sg":
    inputs = {rel_in: datasets.sg_forest_edges(np.random.default_rng(seed), case["n"])}
  elif path == "tc_batch":
    rows, bounds = batch.pack(_batch_instances(case, seed))
    inputs = {rel_in: rows}
  elif path == "andersen":
    d = case["div"]
    inputs = datasets.andersen_inputs(seed, n_vars=200_000 // d, n_objs=50_000 // d,
                                      sizes=(100_000 // d, 400_000 // d, 100_000 // d, 100_000 // d))
  else:
    inputs = {rel_in: _rmat(case["scale"], case["factor"], seed, path != "reach")}
    if path == "reach":
      # the source: a vertex of the graph's dense corner, so that most of it is reached
      inputs["Src"] = np.random.default_rng(seed).integers(0, 16, size=(1, 1), dtype=np.uint32)
  # the caller's result buffers (rows past the result stay 0)
  cap = _capacity(case)
  return {"path": path, "lib": programs.load(program), "inputs": inputs, "rel": rel_out,
          "bounds": bounds, "rows": np.zeros((cap, arity), np.uint32) if arity else None,
          "deltas": np.zeros(_ITERS * (bounds.size - 1 if bounds is not None else 1), np.uint64),
          "cuts": np.zeros(bounds.size, np.uint64) if bounds is not None else None}


# --------------------------------------------------------------------- run ----
def _u32(a):
  return a.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))


def _u64(a, kind=ctypes.c_uint64):
  return a.ctypes.data_as(ctypes.POINTER(kind))


def _session(s):
  """One whole session into the caller's buffers; returns them."""
  lib, rel = s["lib"], s["rel"].encode()
  if lib.init() != 0:
    raise RuntimeError("srdatalog_init failed")
  try:
    for name, rows in s["inputs"].items():
      lib.load_rows(name, rows)
    if s["bounds"] is not None:
      lib.set_instances(s["bounds"])
    if lib.run(0) != 0:
      raise RuntimeError("srdatalog_run failed")
    if s["rows"] is None:   # a count-only rule
      return {"count": lib.size(s["rel"])}
    n = ctypes.c_uint64()
    out = {"rows": s["rows"], "deltas": s["deltas"]}
    if s["bounds"] is None:
      rc = lib.lib.srdatalog_export(rel, _u32(s["rows"]), s["rows"].shape[0], ctypes.byref(n))
      iters = lib.lib.srdatalog_delta_sizes(rel, _u64(s["deltas"], ctypes.c_ulonglong), _ITERS)
    else:
      out["cuts"] = s["cuts"]
      rc = lib.lib.srdatalog_export_instances(rel, _u32(s["rows"]), s["rows"].shape[0],
                                              ctypes.byref(n), _u64(s["cuts"]))
      iters = lib.lib.srdatalog_instance_delta_sizes(rel, _u64(s["deltas"], ctypes.c_ulonglong),
                                                     _ITERS)
    if rc != 0 or iters < 0:
      raise RuntimeError("export failed")
    out["size"] = n.value
    return out
  finally:
    lib.shutdown()


def run(state):
  if state["path"] != "sort":
    return _session(state)
  s = state
  rc = s["lib"].srd_prim_sort_dedup_noalloc(
      s["cols"].data_ptr(), s["n"], s["n"], s["k"], s["out"].data_ptr(), s["n"],
      s["root_vals"].data_ptr(), s["root_offs"].data_ptr(), s["counts"].data_ptr(),
      torch.cuda.current_stream().cuda_stream)
  if rc != 0:
    raise RuntimeError(s["lib"].srd_last_error().decode())
  return [s["out"], s["root_vals"], s["root_offs"], s["counts"]]


# -------------------------------------------------------- work and checks ----
def _sizes(case):
  """(input words, output words) of one pass.  Result sizes follow the
  generators: measured at a few sizes and interpolated."""
  path = case["path"]
  if path == "sort":
    return case["n"] * case["k"], case["n"] * case["k"]
  if path == "tc":
    return 2 * case["m"], 2 * _closure(case["n"], case["m"] / case["n"])
  if path == "sg":
    return 2 * case["n"], 2 * int(0.45 * case["n"] ** 2)
  if path == "tc_batch":
    n = math.sqrt(case["n_lo"] * case["n_hi"])
    return int(case["count"] * n * 5.5), 2 * case["count"] * _closure(1.2 * n, 2.75)
  if path == "andersen":
    return 1_400_000 // case["div"], 2 * int(24e6 * (10 / case["div"]) ** 1.88)
  edges = 0.93 * case["factor"] * 2 ** case["scale"]
  if path == "reach":
    return int(2 * edges), int(0.6 * 2 ** case["scale"])
  tri = 0.9 * edges * case["factor"] * 2 ** (0.12 * (case["scale"] - 14))
  return int(2 * edges), int(3 * tri) if path == "triangle" else 2


def _closure(n, d):
  """Expected pairs of a closure of n vertices at mean out-degree d: the
  share s of vertices that reach (are reached by) most others solves
  s = 1 - exp(-d s)."""
  s = 1.0
  for _ in range(50):
    s = 1 - math.exp(-d * s)
  return int((s * n) ** 2)


def _capacity(case):
  """Rows of the caller's result buffer: bounds of the result's size."""
  if case["path"] in ("tc", "sg"):
    return case["n"] ** 2
  if case["path"] == "tc_batch":
    return case["count"] * case["n_hi"] ** 2
  if case["path"] == "reach":
    return 1 << case["scale"]
  if case["path"] == "andersen":
    return _sizes(case)[1]
  return _sizes(case)[1] + 100_000


def work(case):
  a, b = _sizes(case)
  return {"bytes": 4 * (a + b), "flops": 0}


def tolerance(case):
  return "exact"


def _exact_sort(case, seed):
  cols = _sort_columns(case, seed).cpu().numpy().view(np.uint32)
  k, n = cols.shape
  order = np.lexsort(cols[::-1])
  s = cols[:, order]
  first = np.ones(n, dtype=bool)
  first[1:] = (s[:, 1:] != s[:, :-1]).any(axis=0)
  s = s[:, first]
  u = s.shape[1]
  head = np.flatnonzero(np.concatenate([[True], s[0, 1:] != s[0, :-1]]))
  out = np.zeros((k, n), dtype=np.uint32)
  vals, offs = np.zeros(n, dtype=np.uint32), np.zeros(n + 1, dtype=np.uint32)
  out[:, :u] = s
  vals[:head.size], offs[:head.size] = s[0, head], head
  offs[head.size] = u
  return [x.view(np.int32) for x in (out, vals, offs)] + [np.array([u, head.size, 0], dtype=np.int64)]


def _exact_tc(case, seed):
  """Semi-naive closure with boolean matrices held in doubles; iteration 0
  reads the whole closure so far, as the program's fixpoint does."""
  n = case["n"]
  e = torch.from_numpy(datasets.tc_edges(seed, n, case["m"]).astype(np.int64)).cuda()
  a = torch.zeros(n, n, dtype=torch.float64, device="cuda")
  a[e[:, 0], e[:, 1]] = 1
  full = a > 0
  delta, deltas = full, []
  while True:
    delta = ((delta.double() @ a) > 0) & ~full
    full = full | delta
    deltas.append(int(delta.sum()))
    if deltas[-1] == 0:
      break
  rows = full.nonzero().to(torch.int32).cpu().numpy().view(np.uint32)
  return _padded(case, rows, deltas)


def _padded(case, rows, deltas):
  out = {"rows": np.zeros((_capacity(case), rows.shape[1]), np.uint32),
         "deltas": np.zeros(_ITERS, np.uint64), "size": rows.shape[0]}
  out["rows"][:rows.shape[0]] = rows
  out["deltas"][:len(deltas)] = deltas
  return out


def _exact_triangles(case, seed, listing):
  """Every wedge x < y, x < z tested against the edge set."""
  e = torch.from_numpy(_rmat(case["scale"], case["factor"], seed, True).astype(np.int64)).cuda()
  keys = torch.sort((e[:, 0] << 32) | e[:, 1]).values
  u, v = keys >> 32, keys & 0xFFFFFFFF
  lo, hi = torch.searchsorted(u, v), torch.searchsorted(u, v, right=True)
  out, total = [], 0
  at, cum = 0, torch.cumsum(hi - lo, 0)
  while at < keys.numel():
    done = int(cum[at - 1]) if at else 0
    to = max(at + 1, int(torch.searchsorted(cum, done + (1 << 27))))
    cnt = hi[at:to] - lo[at:to]
    idx = torch.repeat_interleave(torch.arange(at, to, device="cuda"), cnt)
    z = v[lo[idx] + torch.arange(idx.numel(), device="cuda") -
          torch.repeat_interleave(torch.cumsum(cnt, 0) - cnt, cnt)]
    want = (u[idx] << 32) | z
    pos = torch.searchsorted(keys, want).clamp(max=keys.numel() - 1)
    hit = keys[pos] == want
    total += int(hit.sum())
    if listing:
      out.append(torch.stack([u[idx][hit], v[idx][hit], z[hit]], dim=1).to(torch.int32).cpu().numpy())
    at = to
  if not listing:
    return {"count": total}
  rows = np.concatenate(out).view(np.uint32)
  return _padded(case, rows, [rows.shape[0]])


def exact(case, seed):
  path = case["path"]
  if path == "sort":
    return _exact_sort(case, seed)
  if path == "tc":
    return _exact_tc(case, seed)
  if path == "triangle" or (path == "triangle_count" and case["scale"] <= 17):
    return _exact_triangles(case, seed, path == "triangle")
  return None   # no restatement in plain torch finishes in seconds
