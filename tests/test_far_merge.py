"""The far field's merged own-side fragments (sym_geometry.hpp), checked on the
host by tests/cpp/far_merge_check: what far_kernel's workgroups write is what
the combine reads, each fragment once and in order.  No GPU involved."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "cpp", "far_merge_check")


@pytest.mark.skipif(not os.path.exists(EXE), reason="tests/cpp/far_merge_check not built (run __graft_entry__.build())")
def test_combine_reads_what_the_far_field_writes():
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok ")
