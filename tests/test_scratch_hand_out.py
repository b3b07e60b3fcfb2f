"""CPU: two host threads with a stream each never hand partial sums over through the same scratch (tests/cpp/scratch_hand_out.cpp, which
stands in for the HIP runtime)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_two_threads_are_never_given_the_same_scratch():
    sys.path.insert(0, os.path.join(ROOT, "tests", "cpp"))
    import build_host_tests as b

    if not os.path.exists(b.SCRATCH_BIN):
        import oracle  # noqa: F401  (builds the checker that the other host tests link against)

        b.build_host_tests()
    res = subprocess.run([b.SCRATCH_BIN], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and "scratch hand-out ok" in res.stdout, res.stdout + res.stderr
