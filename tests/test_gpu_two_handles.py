"""Handles in use on several threads at once: the exact relax-6 sweeps with the
vector in LDS, on levels of different sizes that share one kernel."""
import threading

import numpy as np
import pytest

import jxpamg_all_amd as jx
from tests.test_gpu_lds_sweep import level
from tests.test_gpu_rowgroup import dev, host, trivial_bsr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("prec", [0, 1])
def test_exact_sweeps_of_two_sizes_at_once(prec):
    sizes = (200, 20000, 900, 15000)
    jobs = []
    for n in sizes:
        ia, ja, a = level(n, 6, n)
        s = jx.Solver(trivial_bsr(n), jx.Hierarchy([(ia, ja, a, n)], []), jx.default_params(precond_precision=prec))
        rng = np.random.default_rng(n)
        jobs.append((s, dev(rng.standard_normal(n)), dev(rng.standard_normal(n))))
    torch.cuda.synchronize()

    def sweeps(k, out, calls=30):
        s, f, u0 = jobs[k]
        u = u0.clone()
        torch.cuda.current_stream().synchronize()
        for _ in range(calls):
            s.hsgs(0, f.data_ptr(), u.data_ptr())
        out[k] = u

    alone, together = {}, {}
    for k in range(len(sizes)):
        sweeps(k, alone)
    print(f"[gpu] exact sweeps on {len(sizes)} threads precision {prec}", flush=True)
    threads = [threading.Thread(target=sweeps, args=(k, together)) for k in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert sorted(together) == list(range(len(sizes)))
    for k in range(len(sizes)):
        assert np.array_equal(host(together[k]), host(alone[k]))
        assert np.all(np.isfinite(host(alone[k])))
        jobs[k][0].close()
