"""The stage-2 sweep from the prolongated pressure (one column of each block,
whole blocks only below the row inside its partition) against the oracle: all
block sizes and storages, partitions of one to eight rows, rows of odd and even
slot counts over several batches, the last partial slice, each pressure index."""
import numpy as np
import pytest

import jxpamg_all_amd as jx
from oracle.cpu_ref import Oracle
from tests._common import relerr
from tests.test_gpu_rowgroup import dev, host
from tests.test_gpu_syncfree import block_system

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nb,rowlen", [(1, 0), (65, 4), (640, 7), (1001, 15)])
@pytest.mark.parametrize("b", [2, 3, 4])
def test_first_sweep_vs_oracle(nb, rowlen, b):
    A = block_system(nb, b, rowlen, nb + b)
    r = np.random.default_rng(nb + b).standard_normal(A.n)
    for pidx in (0, b - 1):
        H = jx.amg_setup(*jx.extract_pressure(A, pidx))
        o = Oracle(A, H)
        o.set_relax_threads([min(len(m[0]) - 1, -(-(len(m[0]) - 1) // 4)) for m in H.A])
        for chunk in (1, 2, 4, 7, 8):
            want = o.cpr(r, o.params(stage2_maxit=1, stage2_parts=-(-nb // chunk), pressure_index=pidx))
            for prec, s2p in ((0, 0), (0, 1), (1, 1), (0, 2), (1, 2)):
                print(f"[gpu] first sweep nb {nb} b {b} pidx {pidx} chunk {chunk} prec {prec} blocks {s2p}", flush=True)
                s = jx.Solver(A, H, jx.default_params(relax_chunk=4, stage2_chunk=chunk, stage2_maxit=1,
                                                      pressure_index=pidx, precond_precision=prec,
                                                      stage2_precision=s2p))
                x = dev(np.zeros(A.n))
                s.precond(dev(r).data_ptr(), x.data_ptr())
                # as for the other partitioned sweeps: FP64, FP32 and FP16 blocks
                assert relerr(host(x), want) < (1e-9, 2e-5, 5e-3)[s2p]
                s.close()
