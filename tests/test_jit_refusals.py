"""What a refused specialised launch rules out (clexmc_jit.h, compiled for the
host in tests/cpp/jit_refusals_check): after the spread kernel, only that kernel
of that kind, so that the ordinary specialised kernel, which takes less LDS, is
tried next; after the ordinary kernel, launches with as much LDS or more."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHECK = os.path.join(ROOT, "tests", "cpp", "jit_refusals_check")


@pytest.mark.skipif(not os.path.exists(CHECK), reason="tests/cpp/jit_refusals_check not built (run build())")
def test_refusals_rule_out_no_smaller_launch():
    out = subprocess.run([CHECK], capture_output=True, text=True, check=True).stdout.splitlines()
    got = {l.split()[0]: [int(x) for x in l.split()[2::2]] for l in out}
    assert got == {"start": [1, 1, 1, 1, 1], "spread": [1, 0, 1, 1, 1], "ordinary": [1, 0, 1, 0, 0],
                   "larger": [1, 0, 1, 0, 0]}
