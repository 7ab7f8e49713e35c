"""The team of host threads that copies the caller's arrays (no GPU): whole copies, and forked processes
that hold a team whose threads they do not have.  Runs tests/native/host_io_check."""
import subprocess
from pathlib import Path

import pytest

CHECK = Path(__file__).resolve().parent / "native" / "host_io_check"


def test_copy_team():
    if not CHECK.exists():
        pytest.fail("tests/native/host_io_check is not built (run __graft_entry__.build())")
    p = subprocess.run([str(CHECK)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    print(p.stdout)
    assert p.returncode == 0 and "host_io_check: OK" in p.stdout
