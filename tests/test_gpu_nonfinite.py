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
from tests.test_gpu_syncfree import block_system

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


def faulty_blocks(nb, b, rowlen, pidx, value, where, chunk):
    """a system with one such value outside column pidx of a block that
    couples two partitions (where 0), or lies above (1) or below (2) the
    diagonal inside one; and the row"""
    A = block_system(nb, b, rowlen, nb + b)
    T = -(-nb // chunk)
    part = np.repeat(np.arange(T), [len(p) for p in np.array_split(np.arange(nb), T)])
    rows = np.repeat(np.arange(nb), np.diff(A.ia))
    inside = part[rows] == part[A.ja]
    at = np.nonzero([~inside, inside & (A.ja > rows), inside & (A.ja < rows)][where])[0]
    k = int(at[len(at) // 2])
    A.a.reshape(-1, b, b)[k, 0, (pidx + 1) % b] = value
    return A, int(rows[k])


@pytest.mark.parametrize("b", [2, 3, 4])
@pytest.mark.parametrize("value", [np.inf, np.nan, 1e300])
@pytest.mark.parametrize("prec,s2p", [(0, 0), (1, 1), (0, 1), (1, 2)])
def test_first_stage2_sweep_nonfinite_block(b, value, prec, s2p):
    """the sweep from the prolongated pressure, whose other unknowns are zeros"""
    nb, chunk = 700, 4
    for where in range(3):
        for pidx in (0, b - 1):
            A, row = faulty_blocks(nb, b, 7, pidx, value, where, chunk)
            H = jx.amg_setup(*jx.extract_pressure(A, pidx))
            s = jx.Solver(A, H, jx.default_params(relax_chunk=4, stage2_chunk=chunk, stage2_maxit=1,
                                                  pressure_index=pidx, precond_precision=prec, stage2_precision=s2p))
            r = np.random.default_rng(b).standard_normal(A.n)
            x = dev(np.zeros(A.n))
            print(f"[gpu] first sweep b {b} value {value} where {where} pidx {pidx} prec {prec} blocks {s2p}", flush=True)
            s.precond(dev(r).data_ptr(), x.data_ptr())
            got = kinds(host(x)).reshape(nb, b)
            s.close()
            if value == 1e300 and s2p != 1:
                # finite in FP64; an FP16 row is scaled by its largest value (overflowed scale: only the row's finiteness goes)
                assert s2p == 2 or not got.any()
                continue
            # the value times a zero (below the diagonal: times a new value) in the row, whose
            # inverted diagonal block spreads it over the row's unknowns, then the partition's later rows
            assert np.all(got[row] != 0) and (where == 2 or np.all(got[row] == 2))
            keep = np.ones(nb, bool)
            T = -(-nb // chunk)
            p = [q for q in np.array_split(np.arange(nb), T) if row in q][0]
            keep[p[p >= row]] = False
            assert not got[keep].any()


@pytest.mark.parametrize("value", [-np.inf, np.nan, 1e300])
@pytest.mark.parametrize("rowlen", [6, 40])
@pytest.mark.parametrize("prec", [0, 1])
def test_chunked_zero_guess_nonfinite_coupling(value, rowlen, prec):
    """a chunk's own coupling meets the zeros of the guess: the chunk is NaN, the others are finite"""
    n, chunk = 2000, 4
    ia, ja, a = level(n, rowlen, rowlen)
    rows = np.repeat(np.arange(n), np.diff(ia))
    at = np.nonzero((ja // chunk == rows // chunk) & (ja > rows))[0]
    k = int(at[len(at) // 2])
    a[k] = value
    H = jx.Hierarchy([(ia, ja, a, n)], [])
    A = trivial_bsr(n)
    s = jx.Solver(A, H, jx.default_params(relax_chunk=chunk, precond_precision=prec, stage2_maxit=0))
    r = np.random.default_rng(rowlen).standard_normal(A.n)
    x = dev(np.zeros(A.n))
    print(f"[gpu] zero guess value {value} mean row {len(ja) / n:.1f} precision {prec}", flush=True)
    s.precond(dev(r).data_ptr(), x.data_ptr())
    got = kinds(host(x)).reshape(n, 2)[:, 0]
    want = np.zeros(n, int)
    if value != 1e300 or prec:
        want[rows[k] // chunk * chunk:][:chunk] = 2
    assert np.array_equal(got, want)
    s.close()
