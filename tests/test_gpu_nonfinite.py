"""Infinite and NaN matrix entries: they reach the entries of a result that the
arithmetic takes them to (an infinite coupling leaves an infinite value, an
entry that meets a zero of the vector a NaN), in the kernels that skip terms
as in the general ones."""
import numpy as np
import pytest

import jxpamg_all_amd as jx
from oracle.cpu_ref import Oracle
from tests.test_gpu_lds_sweep import level
from tests.test_gpu_rowgroup import dev, host, trivial_bsr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def kinds(x):
    """0 finite, 1 infinite, 2 NaN"""
    return np.where(np.isnan(x), 2, np.where(np.isinf(x), 1, 0))


@pytest.mark.parametrize("n,rowlen,symmetric", [(300, 6, False), (300, 40, False), (21000, 6, True), (300, 6, True)])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("upper", [False, True])
def test_exact_sweep_infinite_coupling(n, rowlen, symmetric, prec, upper):
    """one lane per row, row groups, and (small symmetric levels) the vector in LDS"""
    ia, ja, a = level(n, rowlen, 5 * n + rowlen, symmetric)
    rows = np.repeat(np.arange(n), np.diff(ia))
    a[np.nonzero(ja > rows if upper else ja < rows)[0][-3]] = -np.inf
    H = jx.Hierarchy([(ia, ja, a, n)], [])
    A = trivial_bsr(n)
    print(f"[gpu] infinite coupling n {n} mean row {len(ja) / n:.1f} symmetric {symmetric} precision {prec} "
          f"upper {upper}", flush=True)
    rng = np.random.default_rng(n)
    f, u0 = rng.standard_normal(n), rng.standard_normal(n)
    s = jx.Solver(A, H, jx.default_params(precond_precision=prec))
    d_u = dev(u0)
    s.hsgs(0, dev(f).data_ptr(), d_u.data_ptr())
    with np.errstate(invalid="ignore"):
        want = kinds(Oracle(A, H).relax6(0, f, u0))
    assert 0 < np.count_nonzero(want) and np.array_equal(kinds(host(d_u)), want)
    s.close()
