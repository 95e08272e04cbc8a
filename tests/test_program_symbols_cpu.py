"""A program library resolves its generated launchers and kernels to its own,
whatever other programs the process has loaded: no relocation is left that
names one (two programs with a rule of the same name at the same place define
the same names)."""
import os
import subprocess

import pytest

from srdatalog_hip import programs


@pytest.mark.parametrize("name", sorted(programs.PROGRAMS))
def test_no_generated_symbol_is_bound_at_load(name):
  path = programs.so_path(name)
  if not os.path.exists(path):
    pytest.skip("libraries not built (run __graft_entry__.build())")
  out = subprocess.run(["readelf", "-Wr", path], capture_output=True, text=True, check=True).stdout
  assert "srd_engine_create_ext" in out          # what does come from the runtime
  assert not [line for line in out.splitlines() if "srdp_" in line]
