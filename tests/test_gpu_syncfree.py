"""Sync-free sweeps whose results are their own flags (exact relax 6, the
one-rank stage 2, BILU(0) solves) against the oracle: single slices, remainders,
rows over several batches of entries, all block sizes, and inputs that hold
the very bits a result not yet written holds."""
import numpy as np
import pytest

import jxpamg_all_amd as jx
from oracle.cpu_ref import Oracle
from tests._common import relerr
from tests.test_gpu_lds_sweep import level
from tests.test_gpu_rowgroup import dev, host, trivial_bsr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ARMED = 0x7FF4A5A5A5A5A5A5  # what a double of a launch in progress holds


def armed_at(x, k):
    """x on the device with entry k holding the armed bits"""
    v = np.ascontiguousarray(x, np.float64).view(np.int64).copy()
    v[k] = ARMED
    return torch.tensor(v, device="cuda").view(torch.float64)


def block_system(nb, b, rowlen, seed):
    """block-diagonally dominant, symmetric pattern, rows sorted behind the diagonal"""
    ia, ja, _ = level(nb, rowlen, seed)
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1.0, 1.0, (len(ja), b, b))
    for i in range(nb):
        ja[ia[i] + 1:ia[i + 1]] = np.sort(ja[ia[i] + 1:ia[i + 1]])
        a[ia[i]] += np.eye(b) * (1.1 * b * (ia[i + 1] - ia[i]))
    return jx.BSRMatrix(nb, b, ia, ja, a.ravel())


@pytest.mark.parametrize("nb,rowlen", [(1, 0), (64, 6), (65, 3), (700, 7), (1500, 22)])
@pytest.mark.parametrize("b", [2, 3, 4])
def test_stage2_and_bilu_vs_oracle(nb, rowlen, b):
    A = block_system(nb, b, rowlen, 100 * nb + b)
    H = jx.amg_setup(*jx.extract_pressure(A))
    o = Oracle(A, H)
    print(f"[gpu] sync-free stage 2 nb {nb} b {b} mean row {len(A.ja) / nb:.1f}", flush=True)
    rng = np.random.default_rng(b)
    r, x0 = rng.standard_normal(A.n), rng.standard_normal(A.n)
    s = jx.Solver(A, H, jx.default_params())
    x = dev(x0)
    s.bhgs(x.data_ptr(), dev(r).data_ptr(), 0.7, 0.9)
    assert relerr(host(x), o.bhgs(x0, r)) < 1e-11
    x = dev(np.zeros(A.n))
    s.precond(dev(r).data_ptr(), x.data_ptr())
    assert relerr(host(x), o.cpr(r, o.params())) < 1e-9
    assert s.error_flag() == 0
    s.close()
    for s2p in (0, 1, 2):
        s = jx.Solver(A, H, jx.default_params(stage2_solver_type=5, stage2_precision=s2p))
        z, d_r = dev(np.zeros(A.n)), dev(r)
        s.bilu_solve(d_r.data_ptr(), z.data_ptr())
        assert relerr(host(z), o.bilu0_solve(r)) < (1e-11, 1e-5, 1e-2)[s2p]
        # the armed bits as an input are one NaN among others
        d_r = armed_at(r, A.n // 2)
        s.bilu_solve(d_r.data_ptr(), z.data_ptr())
        assert np.isnan(host(z)[A.n // 2]) and s.error_flag() == 0
        s.close()


@pytest.mark.parametrize("rowlen,zero_every", [(6, 0), (7, 5), (11, 0), (24, 0), (90, 0)])
@pytest.mark.parametrize("prec", [0, 1, 2])
def test_exact_sweep_vs_oracle(rowlen, zero_every, prec):
    n = 41000 if rowlen < 12 else 4000
    # an unsymmetric pattern keeps the small levels out of LDS
    ia, ja, a = level(n, rowlen, 7 * rowlen, n > 40961, zero_every)
    H = jx.Hierarchy([(ia, ja, a, n)], [])
    A = trivial_bsr(n)
    print(f"[gpu] sync-free sweep n {n} mean row {len(ja) / n:.1f} precision {prec}", flush=True)
    rng = np.random.default_rng(rowlen)
    f, u0 = rng.standard_normal(n), rng.standard_normal(n)
    s = jx.Solver(A, H, jx.default_params(precond_precision=prec))
    d_f, d_u = dev(f), dev(u0)
    s.hsgs(0, d_f.data_ptr(), d_u.data_ptr())
    # FP32: entries and sums rounded to 24 bits; FP16: entries to 11
    assert relerr(host(d_u), Oracle(A, H).relax6(0, f, u0)) < (1e-11, 2e-5, 1e-2)[prec]
    d_u = armed_at(u0, n - 1)
    s.hsgs(0, d_f.data_ptr(), d_u.data_ptr())
    host(d_u)
    assert s.error_flag() == 0
    s.close()
