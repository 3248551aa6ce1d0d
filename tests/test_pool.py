"""The library's block pool over an allocator that counts and can run out
(oracle/pool_check.cpp, under ThreadSanitizer): reuse and its bound, idle
blocks that go back to other pools and to plain allocations where memory runs
out, failing allocations of the pool's own records, and blocks that other
threads give back.

CPU only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
POOL = os.path.join(ROOT, "oracle", "pool_check")


def test_pool_gives_back_what_it_keeps():
    if not os.path.exists(POOL):
        pytest.fail(f"{POOL} is not built; run `make -C oracle`")
    r = subprocess.run([POOL], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-4000:]
    assert r.stdout.split() == ["ok"] * 5
