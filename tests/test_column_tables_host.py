"""The column kernel's host tables under the address and undefined-behaviour sanitizers:
every item, entry and string record walked as the kernel walks it, against the row-by-row
sum (tests/cpp/test_column_tables.cpp).  Host code only: no GPU."""

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
BIN = os.path.join(HERE, "cpp", "test_column_tables")


def test_column_tables_sanitized():
    if not os.path.exists(BIN):
        sys.path.insert(0, os.path.join(os.path.dirname(HERE), "fast-pauli_amd"))
        import build as B

        B.build_tile_test("test_column_tables")
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0", UBSAN_OPTIONS="print_stacktrace=1")
    p = subprocess.run([BIN], capture_output=True, text=True, timeout=300, env=env)
    assert p.returncode == 0, p.stdout + p.stderr
    assert " 0 failures" in p.stdout, p.stdout
