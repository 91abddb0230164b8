"""GPU parity on both sides of the line between launches with few bytes of
arguments and the general ones: fused rank 4 and 5 of tiles, 8 MiB moved, 5 and
6 row dimensions, 2^20 vectors of rows, with partial tiles, padding and
misaligned pointers; bit-exact against the oracle."""
import pytest

from common import CODE
from test_gpu_parity import check

pytestmark = pytest.mark.gpu

TILES = [  # perm, size
    ([1, 0], [1024, 1024]), ([1, 0], [1031, 1024]), ([1, 0], [1, 4099]), ([1, 0], [2053, 3]),
    ([2, 0, 1], [67, 5, 131]), ([2, 0, 3, 1], [37, 21, 19, 5]), ([3, 2, 1, 0], [33, 17, 9, 23]),
    ([3, 0, 2, 1], [5, 130, 2, 41]), ([4, 2, 0, 3, 1], [11, 7, 5, 9, 13]), ([4, 3, 2, 1, 0], [12, 4, 10, 6, 9]),
]
ROWS = [
    ([0, 2, 1], [16, 300, 218]), ([0, 2, 1], [16, 300, 219]), ([0, 3, 2, 1], [9, 7, 11, 5]),
    ([0, 5, 4, 3, 2, 1], [6, 3, 5, 4, 7, 2]), ([0, 6, 5, 4, 3, 2, 1], [5, 3, 2, 4, 3, 2, 5]),
    ([0, 2, 1], [4, 2048, 511]), ([0, 2, 1], [4, 2048, 512]),
]


@pytest.mark.parametrize("code", ["s", "d", "c", "z", "b", "sb", "ds"])
def test_tiles_on_both_sides(gpu, code):
    tA, tB = CODE[code]
    for n, (perm, size) in enumerate(TILES):
        for beta in (0.0, 0.75):
            check(gpu, tA, tB, perm, size, 1.25, beta, seed=n)
        lda, ldb = [s + 2 for s in size], [size[p] + 1 for p in perm]
        check(gpu, tA, tB, perm, size, 1.25, 0.75, lda, ldb, seed=n)
        check(gpu, tA, tB, perm, size, 1.0, 0.0, seed=n, offset_a=1, offset_b=1)


@pytest.mark.parametrize("code", ["s", "d", "b", "sb"])
def test_rows_on_both_sides(gpu, code):
    tA, tB = CODE[code]
    for n, (perm, size) in enumerate(ROWS):
        for beta in (0.0, 0.75):
            check(gpu, tA, tB, perm, size, 1.25, beta, seed=n)
        check(gpu, tA, tB, perm, size, 1.0, 0.0, seed=n, offset_a=1, offset_b=1)


def test_many_small_rows_fit_the_workspace(gpu):
    """40000 row copies in one allocation-free grouped launch: 336 bytes of
    work table per op is what it held before its records were split."""
    import torch
    from ttc_amd import runtime as rt
    nops, size = 40000, [4, 3, 2]
    A = torch.randn(nops, 24, device=gpu)
    B = torch.zeros(nops, 24, device=gpu)
    a, b = A.data_ptr(), B.data_ptr()
    rt.batch_execute_noalloc([dict(type_a=rt.S, perm=[0, 2, 1], size=size, alpha=1.0, beta=0.0, A=a + 96 * i,
                                   B=b + 96 * i) for i in range(nops)])
    torch.cuda.synchronize()
    assert torch.equal(B.view(nops, 3, 2, 4), A.view(nops, 2, 3, 4).transpose(1, 2))
