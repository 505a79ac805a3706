"""Which kernel form a plan runs with, and sizing for plans whose fields no
call would accept (host logic, no GPU)."""
import os
import subprocess
import sys

import pytest

import segtaco_amd as S

PROBE = """
import sys
sys.path.insert(0, {root!r})
import segtaco_amd as S
A = S.csr_desc(1000, 1000, 5000, 0x1000, 0x2000, 0x3000, S.DT_F32)
p = S.make_plan("eb_cs", vec={vec}, col_lanes={lanes}, group=64, tile=64, comp_threshold=0)
print(S.{call}(A, 64, p))
"""


# In a process of its own: a sizing query must neither hang nor raise a signal.
@pytest.mark.parametrize("call,vec,lanes", [("cs_workspace_layout", 4, 0),
                                            ("cs_workspace_layout", 1, 0),
                                            ("workspace_bytes", -1, 8),
                                            ("workspace_bytes", -2, 8)])
def test_eb_cs_sizing_of_unusual_plans(call, vec, lanes):
    root = os.path.dirname(os.path.dirname(os.path.abspath(S.__file__)))
    r = subprocess.run([sys.executable, "-c", PROBE.format(root=root, call=call, vec=vec,
                                                           lanes=lanes)],
                       capture_output=True, text=True, timeout=20)
    assert r.returncode == 0, (r.returncode, r.stderr)
    if call == "cs_workspace_layout":
        A = S.csr_desc(1000, 1000, 5000, 0x1000, 0x2000, 0x3000, S.DT_F32)
        full = S.make_plan("eb_cs", vec=vec, col_lanes=8, group=64, tile=64, comp_threshold=0)
        assert r.stdout.strip() == str(S.cs_workspace_layout(A, 64, full))
