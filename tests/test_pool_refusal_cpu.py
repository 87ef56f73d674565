"""Worker threads that cannot be started: the size is refused where it is
asked for, overlapping calls then work serially, and neither tries again on
every call."""
import subprocess
import sys

from tests import conftest


def test_threads_that_cannot_be_started():
    # a process of its own: the check holds its address space for a moment
    code = "from tests import oracle_lib; print(oracle_lib.load().oracle_pool_refusal())"
    r = subprocess.run([sys.executable, "-c", code], cwd=conftest.ROOT, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0 and r.stdout.split()[-1] == "0", (r.stdout, r.stderr)
