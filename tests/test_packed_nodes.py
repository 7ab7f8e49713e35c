"""The packed nodes on the host (no GPU): leaves placed once each, planes outside the built ones, and
the packed test accepting every ray and interval that the built boxes accept.  Runs
tests/native/packed_check."""
import subprocess
from pathlib import Path

import pytest

CHECK = Path(__file__).resolve().parent / "native" / "packed_check"


@pytest.mark.parametrize("args", [("tree", "4000", "1", "4"), ("tree", "900", "2", "16"), ("tree", "300", "3", "1"),
                                  ("tree", "1", "4", "4"), ("nodes", "5"), ("nodes", "6")])
def test_packed_nodes(args):
    if not CHECK.exists():
        pytest.fail("tests/native/packed_check is not built (run __graft_entry__.build())")
    p = subprocess.run([str(CHECK), *args], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(p.stdout)
    assert p.returncode == 0 and "packed_check: OK" in p.stdout
