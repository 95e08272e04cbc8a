"""__graft_entry__.build() compiles the product alone: a tree whose tests are
missing, or belong to another revision, builds."""
import os
import shutil
import subprocess
import sys

from conftest import ROOT

# the compilers' outputs are not what is tested here: every compile succeeds
STUB = """
import subprocess, sys
sys.path.insert(0, sys.argv[1])
import __graft_entry__ as g
from srdatalog_hip import native, programs
import oracle
done = []
native.build_runtime = lambda *a, **k: done.append("runtime")
oracle.build = lambda *a, **k: done.append("oracle")
programs.build_all = lambda *a, **k: done.append("programs")
g.build()
print(",".join(done))
"""


def test_build_needs_no_tests_folder(tmp_path):
  for d in ("srdatalog-python_amd", "oracle", "include"):
    shutil.copytree(os.path.join(ROOT, d), tmp_path / d,
                    ignore=shutil.ignore_patterns("*.so", "__pycache__", "_lib"))
  shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), tmp_path)
  r = subprocess.run([sys.executable, "-c", STUB, str(tmp_path)], cwd=tmp_path,
                     capture_output=True, text=True, timeout=300)
  assert r.returncode == 0, r.stderr
  assert r.stdout.strip().split(",") == ["runtime", "oracle", "programs"]
