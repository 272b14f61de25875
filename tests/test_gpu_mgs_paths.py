"""The one-launch Arnoldi step against one launch per projection, an
independent path (arnoldi_kernel 1), at the sizes where its tile and number of
workgroups change; and, on vectors that take several workgroups, the ordinary
against the cooperative launch, the speculative start, and a wait that gives up."""
import ctypes

import numpy as np
import pytest

import jxpamg_all_amd as jx
from tests._common import relerr
from tests.test_gpu_rowgroup import dev
from tests.test_gpu_syncfree import block_system

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SEVERAL = 9001  # block rows of two unknowns: 18002 entries, more than one workgroup holds


def solver(nb, **kw):
    A = block_system(nb, 2, 6 if nb > 1 else 0, nb)
    H = jx.Hierarchy([jx.extract_pressure(A) + (nb,)], [])
    return A, jx.Solver(A, H, jx.default_params(**dict(dict(tol=1e-10, relax_chunk=4, stage2_chunk=4), **kw)))


@pytest.mark.parametrize("nb", [1, 2047, 2048, 2049, 4096, 4097, 8192, 8193, SEVERAL, 40000])
def test_step_vs_one_launch_per_projection(nb):
    got = {}
    for kernel in (1, 2, 0):
        A, s = solver(nb, arnoldi_kernel=kernel)
        b = np.random.default_rng(nb).standard_normal(A.n)
        print(f"[gpu] Arnoldi kernel {kernel} n {A.n}", flush=True)
        x, st, hist = s.solve(b)
        assert st.converged == 1 and s.error_flag() == 0
        got[kernel] = (x, st.iterations, hist)
        s.close()
    for kernel in (2, 0):
        # the sums are added in another order: rounding of some ten projections of 80000 entries
        assert got[kernel][1] == got[1][1] and relerr(got[kernel][0], got[1][0]) < 1e-9
        assert relerr(got[kernel][2], got[1][2]) < 1e-11
    # one kernel by two kinds of launch
    assert np.array_equal(got[0][0], got[2][0]) and np.array_equal(got[0][2], got[2][2])


def test_speculative_start_across_workgroups():
    """an unprofiled solve runs a step ahead, a profiled one does not: bit for bit the same"""
    A, s = solver(SEVERAL)
    b = np.random.default_rng(1).standard_normal(A.n)
    x0, st0, h0 = s.solve(b)
    s.profile(True)
    x1, st1, h1 = s.solve(b)
    s.profile(False)
    x2, st2, h2 = s.solve(b)
    assert st0.converged == 1 and s.error_flag() == 0
    assert np.array_equal(h0, h1) and np.array_equal(x0, x1)
    assert np.array_equal(h0, h2) and np.array_equal(x0, x2)
    s.close()


@pytest.mark.parametrize("nb", [SEVERAL, 40000])
def test_wait_that_gives_up_is_reported_and_cleared(nb):
    """A spin limit of zero from the host: a waiting workgroup gives up at its
    first poll and every kernel still exits.  The solve reports it, and the
    next one with the usual limit is a fresh solver's bit for bit."""
    A, s = solver(nb, max_iter=8)
    b = np.random.default_rng(nb).standard_normal(A.n)
    s.set_spin_limit(0)
    d_x, hist, st = dev(np.zeros(A.n)), np.zeros(9), jx.Stats()
    d_b = dev(b)
    print(f"[gpu] forced give-up n {A.n}", flush=True)
    rc = s._L.jxamd_solver_solve_device(s._s, d_b.data_ptr(), d_x.data_ptr(), jx._p(hist), ctypes.byref(st))
    assert rc == 1 and s.error_flag() == 0
    s.set_spin_limit(1 << 24)
    x, _, h = s.solve(b)
    A, fresh = solver(nb, max_iter=8)
    x2, _, h2 = fresh.solve(b)
    assert s.error_flag() == 0 and np.array_equal(x, x2) and np.array_equal(h, h2)
    s.close()
    fresh.close()
