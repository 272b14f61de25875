"""The layouts of the one-workgroup relax-6 sweeps (levels, slices, records,
padding) and of the chunked sweeps from a zero guess, walked on the host under
AddressSanitizer/UBSan as the kernels walk them, against the recurrence."""
import os
import re
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "hoststub")


@pytest.fixture(scope="module")
def driver():
    r = subprocess.run(["make", "-s", "-C", HERE], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return os.path.join(HERE, "_build", "drive_sweeps")


@pytest.mark.parametrize("n,rowlen,symmetric,zero_every", [
    (1, 0, 1, 0), (5, 3, 1, 0), (64, 6, 1, 0), (65, 6, 1, 7), (700, 40, 1, 0), (3000, 7, 1, 5), (500, 300, 1, 0),
    (1100, 5, 1, 0), (2500, 24, 0, 0), (20479, 6, 1, 0), (20480, 6, 1, 0)])
def test_layouts_give_the_recurrence(driver, n, rowlen, symmetric, zero_every):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0", UBSAN_OPTIONS="halt_on_error=1")
    r = subprocess.run([driver, *(str(v) for v in (n, rowlen, symmetric, zero_every))], capture_output=True, text=True,
                       env=env, timeout=300)
    assert r.returncode == 0 and "runtime error" not in r.stderr, r.stdout[-2000:] + r.stderr[-4000:]
    # FP64 and FP32, from zeros and from a vector; 20480 doubles and a padding entry exceed the LDS
    exact = int(re.search(r"exact (\d+)", r.stdout).group(1))
    # (chunks of a whole level are exact calls, too)
    assert exact == 0 if not symmetric else exact >= (2 if n == 20480 else 4)
