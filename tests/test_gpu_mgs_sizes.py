"""Arnoldi steps of vectors around the sizes where the one-launch step changes
its tile and takes a second workgroup, against one launch per projection."""
import numpy as np
import pytest

import jxpamg_all_amd as jx
from tests._common import relerr
from tests.test_gpu_syncfree import block_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2048, 2049, 4096, 4097, 8192, 8193])
def test_one_launch_step_vs_projections(nb):
    A = block_system(nb, 2, 6 if nb > 1 else 0, nb)
    H = jx.amg_setup(*jx.extract_pressure(A))
    b = np.random.default_rng(nb).standard_normal(A.n)
    got = []
    for kernel in (2, 0):
        print(f"[gpu] Arnoldi kernel {kernel} n {A.n}", flush=True)
        s = jx.Solver(A, H, jx.default_params(tol=1e-10, relax_chunk=4, stage2_chunk=4, arnoldi_kernel=kernel))
        x, st, hist = s.solve(b)
        assert st.converged == 1 and s.error_flag() == 0
        got.append((x, st.iterations))
        s.close()
    # the sums are added in another order: rounding of the projections
    assert got[0][1] == got[1][1] and relerr(got[0][0], got[1][0]) < 1e-9
