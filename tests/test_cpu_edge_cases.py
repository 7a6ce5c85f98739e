"""Edge cases of the C ABI on the CPU kernel emulator, under AddressSanitizer
and UndefinedBehaviorSanitizer (tests/cpu_emu/edge_test.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emu")


@pytest.fixture(scope="module")
def edge_test():
    jobs = str(max(1, min(8, os.cpu_count() or 1)))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU], check=True, timeout=1200)
    return os.path.join(EMU, "_build", "edge_test")


@pytest.mark.parametrize("cases", ["spatial centre", "spatial overflow", "autotune", "refused launch", "memory pool", "scratch",
                                   "order of small"])
def test_edge_cases(edge_test, cases):
    r = subprocess.run([edge_test, cases], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and " ok\n" in r.stdout and "ALL OK" in r.stdout, \
        "%s:\n%s\n%s" % (cases, r.stdout[-3000:], r.stderr[-6000:])
