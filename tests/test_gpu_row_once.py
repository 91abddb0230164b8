"""GPU parity of the row copy with one chunk per work-group at the row
lengths where its unaligned vectors can go wrong: rows shorter than, equal to
and just past a vector, odd rows, one chunk and several, padded leading
dimensions and misaligned pointers; bit-exact against the oracle."""
import numpy as np
import pytest

from common import BF16, CODE, F16, S, same_bits, to_device
from oracle import oracle as orc
from test_gpu_cast_batch import E4M3, E5M2, _heavy_input
from test_gpu_parity import check

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 33, 127, 129]


@pytest.mark.parametrize("code", ["s", "d", "c", "z", "b", "h", "sb", "bs", "sd", "ds", "cz"])
def test_row_lengths(gpu, code):
    tA, tB = CODE[code]
    for n0 in ROWS:
        for pad in (0, 3):
            size = [n0, 13, 22]
            lda = [n0 + pad, 13, 22 + pad] if pad else None
            ldb = [n0 + pad + 1, 22 + pad, 13] if pad else None
            for beta in (0.0, 0.75):
                check(gpu, tA, tB, [0, 2, 1], size, 1.25, beta, lda, ldb, seed=n0)
        check(gpu, tA, tB, [0, 2, 1], [n0, 13, 22], 1.0, 0.0, seed=n0, offset_a=1, offset_b=1)


@pytest.mark.parametrize("tA,tB", [(S, E4M3), (BF16, E4M3), (F16, E5M2)])
def test_row_lengths_fp8(gpu, tA, tB):
    import torch
    from ttc_amd import runtime as rt
    for n0 in ROWS:
        size = [n0, 37, 90]
        n = int(np.prod(size))
        A = _heavy_input(tA, n, n0)
        dA, dB = to_device(A, gpu), torch.zeros(n, dtype=torch.uint8, device=gpu)
        amax = torch.full((1,), -1.0, dtype=torch.float32, device=gpu)
        want = np.zeros(n, np.uint8)
        want_amax = orc.cast_fp8(tA, tB, A, want, 0.5, 3.5, [0, 2, 1], size)
        rt.Plan(tA, tB, [0, 2, 1], size, beta_is_zero=True).execute_fp8(dA, dB, 0.5, scale=3.5, amax_out=amax)
        torch.cuda.synchronize()
        assert same_bits(dB.cpu().numpy(), want) and float(amax.item()) == want_amax, (tA, tB, n0)


@pytest.mark.parametrize("n", [2 ** 31 - 1, 2 ** 31 - 7])
def test_rows_of_almost_2_31_elements(gpu, n):
    """One row whose vectors end within a vector of 2^31: every element, and
    nothing behind the row."""
    import torch
    from ttc_amd import runtime as rt
    A = torch.randn(n, dtype=torch.bfloat16, device=gpu)
    B = torch.full((n + 64,), 3.0, dtype=torch.bfloat16, device=gpu)
    step = 1 << 28
    rt.Plan(BF16, BF16, [0], [n], beta_is_zero=True).execute(A, B, 1.0, 0.0)
    torch.cuda.synchronize()
    assert torch.equal(B[:n], A) and bool((B[n:] == 3.0).all())
    rt.Plan(BF16, BF16, [0], [n]).execute(A, B, 1.0, 0.5)
    torch.cuda.synchronize()
    for i in range(0, n, step):
        a = A[i:min(i + step, n)].float()
        assert torch.equal(B[i:min(i + step, n)], (a + 0.5 * a).to(torch.bfloat16)), i
    assert bool((B[n:] == 3.0).all())
    del B
    Q = torch.full((n + 64,), 7, dtype=torch.uint8, device=gpu)
    amax = torch.zeros(1, device=gpu)
    rt.Plan(BF16, E4M3, [0], [n], beta_is_zero=True).execute_fp8(A, Q, 1.0, scale=32.0, amax_out=amax)
    torch.cuda.synchronize()
    top = 0.0
    for i in range(0, n, step):
        a = A[i:min(i + step, n)].float()
        top = max(top, float(a.abs().max()))
        want = (a * 32.0).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)
        assert torch.equal(Q[i:min(i + step, n)], want), i
    assert bool((Q[n:] == 7).all()) and float(amax) == top


@pytest.mark.parametrize("code", ["s", "d", "c", "b", "h"])
def test_scaling_in_place(gpu, code):
    """An identity permutation whose A is its B: rows that are no whole number
    of vectors, dense and padded, alone, misaligned and in a grouped launch."""
    import torch
    from common import from_device, make_case, oracle_run
    from ttc_amd import runtime as rt
    t, _ = CODE[code]
    for n0 in (3, 9, 127, 100003):
        for size, ld in (([n0], None), ([n0, 41], [n0 + 2, 41])):
            perm = list(range(len(size)))
            for beta in (0.0, 0.5):
                A, _ = make_case(t, t, perm, size, ld, ld, seed=n0)
                want = oracle_run(t, t, A, A, 1.25, beta, perm, size, ld, ld)
                plan = rt.Plan(t, t, perm, size, ld, ld, beta == 0.0)
                for off in (0, A.itemsize):
                    X = torch.zeros(A.nbytes + off, dtype=torch.uint8, device=gpu)
                    X[off:] = to_device(A, gpu)
                    plan.execute(X.data_ptr() + off, X.data_ptr() + off, 1.25, beta)
                    torch.cuda.synchronize()
                    assert same_bits(X[off:].cpu().numpy().view(A.dtype), want), (code, size, ld, beta, off)
                X = to_device(A, gpu)
                rt.Batch([dict(type_a=t, perm=perm, size=size, lda=ld, ldb=ld, alpha=1.25, beta=beta, A=X,
                               B=X)]).execute()
                torch.cuda.synchronize()
                assert same_bits(from_device(X, A), want), (code, size, ld, beta, "grouped")
