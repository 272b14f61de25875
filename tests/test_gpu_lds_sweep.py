"""Exact relax-6 sweeps with the level's vector in LDS (one workgroup) against
the oracle: single slices, remainders, long rows over several records, zero
diagonals, the largest level that fits and the first that does not, and
unsymmetric patterns, whose rows may not be updated in place."""
import numpy as np
import pytest

import jxpamg_all_amd as jx
from oracle.cpu_ref import Oracle
from tests._common import relerr
from tests.test_gpu_rowgroup import dev, host, trivial_bsr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def level(n, rowlen, seed, symmetric=True, zero_every=0):
    """Diagonally dominant CSR, diagonal first, rows in random column order."""
    rng = np.random.default_rng(seed)
    m = max(0, rowlen // 2)
    i = np.repeat(np.arange(n), m)
    j = np.clip(i + rng.integers(-3 * rowlen - 1, 3 * rowlen + 2, len(i)), 0, n - 1)
    pairs = np.stack([i, j], 1)[i != j]
    if symmetric:
        pairs = np.concatenate([pairs, pairs[:, ::-1]])
    pairs = np.unique(pairs, axis=0)
    ia, ja, a = [0], [], []
    by = np.split(pairs[:, 1], np.searchsorted(pairs[:, 0], np.arange(1, n)))
    for r in range(n):
        cols = rng.permutation(by[r])
        vals = -rng.uniform(0.1, 1.0, len(cols))
        d = 1.1 * np.abs(vals).sum() + 0.5
        if zero_every and r % zero_every == 1:
            d = 0.0
        ja += [r] + list(cols)
        a += [d] + list(vals)
        ia.append(len(ja))
    return np.array(ia, np.int32), np.array(ja, np.int32), np.array(a)


@pytest.mark.parametrize("n,rowlen,symmetric,zero_every", [
    (1, 0, True, 0), (5, 3, True, 0), (64, 6, True, 0), (65, 6, True, 7), (700, 40, True, 0), (3000, 7, True, 5),
    (500, 300, True, 0), (2500, 24, False, 0), (20479, 6, True, 0), (20480, 6, True, 0)])
@pytest.mark.parametrize("prec", [0, 1])
def test_exact_sweep_vs_oracle(n, rowlen, symmetric, zero_every, prec):
    ia, ja, a = level(n, rowlen, 11 * n + rowlen, symmetric, zero_every)
    H = jx.Hierarchy([(ia, ja, a, n)], [])
    A = trivial_bsr(n)
    print(f"[gpu] exact sweep n {n} mean row {len(ja) / n:.1f} precision {prec}", flush=True)
    rng = np.random.default_rng(n + prec)
    f, u0 = rng.standard_normal(n), rng.standard_normal(n)
    s = jx.Solver(A, H, jx.default_params(precond_precision=prec))
    d_f, d_u = dev(f), dev(u0)
    s.hsgs(0, d_f.data_ptr(), d_u.data_ptr())
    got = host(d_u)
    # FP32: entries, vectors and sums rounded to 24 bits, as for the other level kernels
    assert relerr(got, Oracle(A, H).relax6(0, f, u0)) < (1e-11 if prec == 0 else 2e-5)
    # an infinite right-hand side spreads to the same entries
    f[n // 2] = np.inf
    d_f, d_u = dev(f), dev(u0)
    s.hsgs(0, d_f.data_ptr(), d_u.data_ptr())
    assert np.array_equal(np.isfinite(host(d_u)), np.isfinite(Oracle(A, H).relax6(0, f, u0)))
    s.close()
