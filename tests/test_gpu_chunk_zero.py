"""Chunked relax 6 from a zero guess (the chunks' own couplings alone) inside
V-cycles against the oracle: chunks of one row to the longest that take this
path and beyond, uneven chunks, partial blocks of 64 chunks, short and long rows."""
import numpy as np
import pytest

import jxpamg_all_amd as jx
from oracle.cpu_ref import Oracle
from tests._common import relerr
from tests.test_gpu_rowgroup import dev, host
from tests.test_gpu_syncfree import block_system

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nb,rowlen", [(1100, 5), (2049, 9), (4000, 30)])
@pytest.mark.parametrize("prec", [0, 1])
def test_chunked_vcycle_vs_oracle(nb, rowlen, prec):
    A = block_system(nb, 2, rowlen, nb)
    H = jx.amg_setup(*jx.extract_pressure(A))
    assert H.num_levels > 1
    f = np.random.default_rng(nb).standard_normal(nb)
    for chunk in (1, 2, 3, 4, 7, 8, 13):
        print(f"[gpu] chunked V-cycle n {nb} mean row {rowlen} chunk {chunk} precision {prec}", flush=True)
        o = Oracle(A, H)
        o.set_relax_threads([min(len(m[0]) - 1, -(-(len(m[0]) - 1) // chunk)) for m in H.A])
        s = jx.Solver(A, H, jx.default_params(relax_chunk=chunk, precond_precision=prec))
        u = dev(np.zeros(nb))
        s.vcycle(dev(f).data_ptr(), u.data_ptr())
        # FP64: summation order; FP32: entries, vectors and sums in 24 bits
        assert relerr(host(u), o.vcycle(f)) < (1e-10 if prec == 0 else 2e-5)
        s.close()
