"""The columns' way between host and device memory (host/column_copy.cpp) on a
stand-in for the runtime: its threads and failures, which no GPU is needed for
(tests/cpp/test_column_copy.cpp)."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.mark.parametrize("name", ["round_trips", "no_memory_for_threads", "copies_after_a_failure",
                                  "threads_that_begin_late", "rings_of_all_handles"])
def test_column_copy(name):
    subprocess.run(["make", "-C", CPP, os.path.join("_build", "test_column_copy")], check=True)
    r = subprocess.run([os.path.join(CPP, "_build", "test_column_copy"), name], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert f"PASS {name}" in r.stdout
