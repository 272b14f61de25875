"""Operations on the assembled arrays at the edges of their dispatches:
True-IMPES coefficients of short, middle and long rows in any column order, and
the residual norm on 8- and 16-byte boundaries, over batches of blocks, and
from more threads than it has work buffers."""
import threading

import numpy as np
import pytest

import jxpamg_all_amd as jx
from tests._common import bits
from tests.test_gpu_lds_sweep import level

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def system(nb, b, rowlen, seed):
    ia, ja, _ = level(nb, rowlen, seed)
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1.0, 1.0, (len(ja), b, b))
    a[ia[:-1]] += 3.0 * np.eye(b)
    return jx.BSRMatrix(nb, b, ia, ja, a.ravel()), rng.standard_normal(nb * b)


@pytest.mark.parametrize("nb,rowlen", [(1, 0), (65, 6), (300, 11), (300, 40)])
@pytest.mark.parametrize("b", [2, 3, 4])
@pytest.mark.parametrize("dtype", [jx.DECOUP_TIMPES, jx.DECOUP_TIMPES2])
def test_true_impes_row_lengths(nb, rowlen, b, dtype):
    A, r = system(nb, b, rowlen, 10 * nb + rowlen)
    want, want_r = jx.decouple(A, r, dtype)
    print(f"[gpu] True-IMPES {dtype} nb {nb} b {b} mean row {len(A.ja) / nb:.1f}", flush=True)
    d = [torch.tensor(v, device="cuda") for v in (A.ia, A.ja, A.a, r)]
    rc = jx.decouple_device(nb, b, *(t.data_ptr() for t in d), dtype, 0, 0, None,
                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert np.array_equal(bits(d[2].cpu().numpy()), bits(want.a))
    assert np.array_equal(bits(d[3].cpu().numpy()), bits(want_r))


@pytest.mark.parametrize("nb,rowlen", [(1, 0), (257, 6), (400, 17)])
@pytest.mark.parametrize("b", [1, 2, 3, 4])
@pytest.mark.parametrize("off", [0, 1])
def test_residual_norm_alignment_and_threads(nb, rowlen, b, off):
    A, r = system(nb, b, rowlen, nb + b)
    x = np.random.default_rng(b).standard_normal(nb * b)
    want = np.array([np.linalg.norm(r - A.to_scipy() @ x), np.linalg.norm(r)])
    print(f"[gpu] residual norm nb {nb} b {b} offset {off}", flush=True)

    def put(v):  # off doubles past a 16-byte boundary
        t = torch.zeros(len(v) + off, dtype=torch.float64, device="cuda")
        t[off:] = torch.tensor(v, device="cuda")
        return t, t.data_ptr() + 8 * off

    d_ia, d_ja = torch.tensor(A.ia, device="cuda"), torch.tensor(A.ja, device="cuda")
    (ta, pa), (tx, px), (tr, pr) = put(A.a), put(x), put(r)
    out = torch.zeros((12, 2), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def call(k):
        for _ in range(3):
            jx.bsr_residual_norm(nb, b, d_ia.data_ptr(), d_ja.data_ptr(), pa, px, pr, out[k].data_ptr())

    call(0)
    threads = [threading.Thread(target=call, args=(k,)) for k in range(1, 12)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    got = out.cpu().numpy()
    assert np.all(bits(got) == bits(got[:1]))
    # sums of at most 17 * 4 products and 1600 squares
    assert np.allclose(got[0], want, rtol=1e-13, atol=0)
