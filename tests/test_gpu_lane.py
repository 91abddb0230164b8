"""GPU parity of the one-tile-per-work-group row x column launch at the tiles
where its walks can go wrong: lanes left over past the last whole column or
row, one lane vector per column, partial last tiles on either group or both,
groups of several dimensions, both instance sizes, every tile numbering and
grid order, one to many tiles, padded tensors; bit-exact against the oracle."""
import pytest

from common import CODE
from test_gpu_parity import check

pytestmark = pytest.mark.gpu

# (perm, size, tile): rows x columns per comment
CASES = [
    ([1, 0], [99, 70], [99, 32]),           # 99 x 32: 58 lanes over, columns 70 = 2 * 32 + 6
    ([1, 0], [300, 40], [250, 4]),          # one column per step, 6 lanes over
    ([1, 0], [40, 300], [4, 250]),          # the mirror image
    ([1, 0], [257, 129], [17, 13]),         # partial on both sides
    ([2, 0, 3, 1], [37, 21, 19, 5], [37, 1, 19, 1]),
    ([3, 1, 0, 2], [12, 10, 9, 11], [12, 3, 1, 5]),   # rows of two dimensions, partial columns
    ([3, 2, 1, 0], [9, 10, 11, 12], [9, 4, 1, 7]),    # both groups end in partial dimensions
    ([1, 0, 2], [33, 65, 20], [33, 13, 3]),           # an extra column dimension
    ([4, 2, 0, 3, 1], [6, 5, 4, 3, 7], [6, 5, 2, 1, 7]),
    ([1, 0], [3, 3], [3, 3]),               # less than one wave
]


@pytest.mark.parametrize("code", ["s", "d", "z", "b", "sb", "bs", "sd", "ds"])
def test_lane_tiles(gpu, code):
    from ttc_amd import runtime as rt
    tA, tB = CODE[code]
    n = 0
    for i, (perm, size, tile) in enumerate(CASES):
        # 16-byte elements take at most 2048 elements per tile, and half the slots of 8-byte ones
        try:
            if not rt.Plan(tA, tB, perm, size, config=dict(family=2, tile=tile, vec_a=1, vec_b=1)).info()["lane_fixed"]:
                continue
        except rt.TTCError:
            continue
        for pad in (0, 1):
            lda = [s + pad * (1 + k % 3) for k, s in enumerate(size)] if pad else None
            ldb = [size[p] + pad * (2 - k % 2) for k, p in enumerate(perm)] if pad else None
            for beta in (0.0, 0.75):
                cfg = dict(family=2, tile=tile, vec_a=1, vec_b=1, tile_order=1 + (i + n) % 4, grid_order=1 + n % 4)
                info = check(gpu, tA, tB, perm, size, 1.25, beta, lda, ldb, seed=n, config=cfg)
                assert info["lane_fixed"] == 1 and info["tile"] == tile, info
                n += 1
    assert n >= 4 * (len(CASES) - (1 if code == "z" else 0))


def test_lane_vector_widths(gpu):
    """Every vector width pair on a full and a partial tile grid."""
    from ttc_amd import runtime as rt
    from ttc_amd.gen_instances import vec_widths
    for code in ("s", "d", "b", "sb", "c"):
        tA, tB = CODE[code]
        for va in vec_widths(rt.DTYPE_BYTES[tA]):
            for vb in vec_widths(rt.DTYPE_BYTES[tB]):
                for size, tile in (([96, 80], [48, 16]), ([104, 88], [64, 48])):
                    for beta in (0.0, 1.5):
                        info = check(gpu, tA, tB, [1, 0], size, 0.5, beta, seed=va + vb,
                                     config=dict(family=2, tile=tile, vec_a=va, vec_b=vb))
                        assert info["lane_fixed"] == 1 and info["vec_a"] == va and info["vec_b"] == vb
