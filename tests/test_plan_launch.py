"""CPU tests of ttc_plan_get_launch: which kernel a plan launches, over how many
tiles or chunks and with how much LDS, beside what ttc_plan_get_info says of the
configuration."""
import pytest

from common import BF16, D, E4M3, S
from ttc_amd import runtime as rt


def launch(tA, tB, perm, size, beta=False, **cfg):
    p = rt.Plan(tA, tB, perm, size, beta_is_zero=not beta, config=cfg or None)
    return p.launch(), p.info()


def test_row_column_tiles():
    tile = [62, 128]
    for order, ids in ((2, 2145), (3, 2376), (4, 2640)):
        one, info = launch(BF16, BF16, [1, 0], [4000, 4100], family=2, tile=tile, vec_a=2, vec_b=2, tile_order=order)
        assert one["kernel"] == rt.KERNEL_TILE and one["units"] == 65 * 33 and info["tiles"] == ids
        assert one["lds_buffers"] == 1 and one["lds_bytes"] < info["lds_bytes"]
        assert one["slots_a"] * one["slot_div"] == info["slots_a"] and one["vec_a"] == 2
        for buffers in (1, 2):
            walk, info = launch(BF16, BF16, [1, 0], [4000, 4100], family=2, tile=tile, vec_a=2, vec_b=2,
                                tile_order=order, lds_buffers=buffers)
            assert walk["kernel"] == rt.KERNEL_TILE_WALK and walk["units"] == ids == info["tiles"]
            assert walk["lds_buffers"] == buffers and walk["lds_bytes"] == info["lds_bytes"] and walk["slot_div"] == 1
            assert walk["lane_fixed"] == 1
    walk, _ = launch(S, S, [1, 0], [4000, 4100], wg_per_cu=2)
    assert walk["kernel"] == rt.KERNEL_TILE_WALK and walk["lane_fixed"] == 0
    small, info = launch(S, S, [1, 0], [300, 200])
    assert small["kernel"] == rt.KERNEL_TILE_SMALL and small["slot_div"] == 2 and small["units"] == info["tiles"]
    cast, _ = launch(BF16, E4M3, [1, 0], [300, 200])
    assert cast["kernel"] == rt.KERNEL_TILE


@pytest.mark.parametrize("tA", [S, D])
def test_full_and_half_instances(tA):
    """slot_div 2 where half the slots cover the tile on both sides."""
    for tile in ([64, 32], [64, 64], [128, 32], [32, 128], [16, 16]):
        try:
            one, info = launch(tA, tA, [1, 0], [4096, 4096], family=2, tile=tile, vec_a=1, vec_b=1)
        except rt.TTCError:
            continue
        half = all(256 // a * (s // 2) >= b for a, b, s in ((tile[0], tile[1], info["slots_a"]),
                                                            (tile[1], tile[0], info["slots_b"])))
        assert one["slot_div"] == (2 if half else 1) and one["units"] == (4096 // tile[0]) * (4096 // tile[1])


def test_row_copies_and_boxes():
    one, _ = launch(S, S, [0, 2, 1], [128, 300, 2000])
    assert one["kernel"] == rt.KERNEL_ROW and one["units"] == 300 * 2000 * 32 // 256 and not one["unaligned"]
    one, info = launch(S, S, [0, 2, 1], [127, 300, 2000])
    assert one["kernel"] == rt.KERNEL_ROW and one["unaligned"] and one["vec_a"] == 4 and info["vec_a"] == 1
    assert one["units"] == -(-300 * 2000 * 32 // 512)
    one, _ = launch(S, S, [0, 2, 1], [127, 30, 20])
    assert one["kernel"] == rt.KERNEL_ROW_SMALL
    one, _ = launch(S, S, [0, 2, 1], [128, 30, 20], family=3, wg_per_cu=4)
    assert one["kernel"] == rt.KERNEL_ROW_WALK and one["slots_a"] == 4
    one, info = launch(S, S, [1, 0], [300, 200], family=1)
    assert one["kernel"] == rt.KERNEL_BOX and one["units"] == info["tiles"] and one["lds_bytes"] == info["lds_bytes"]
    assert launch(S, S, [1, 0], [300, 0])[0]["kernel"] == rt.KERNEL_NONE


@pytest.mark.parametrize("tA,tB,perm,size,beta,kernel", [
    # casts on aligned vectors, from 4 MiB to below 384 MiB moved
    (BF16, E4M3, [0, 2, 1], [128, 100, 100], False, "KERNEL_ROW"),
    (BF16, E4M3, [0, 2, 1], [64, 72, 512], False, "KERNEL_ROW_WALK"),
    (BF16, E4M3, [0, 2, 1], [128, 4096, 255], False, "KERNEL_ROW_WALK"),
    (BF16, E4M3, [0, 2, 1], [128, 4096, 256], False, "KERNEL_ROW"),
    (S, E4M3, [0], [4000000], False, "KERNEL_ROW_WALK"),
    (BF16, E4M3, [0, 2, 1], [127, 300, 121], False, "KERNEL_ROW"),  # unaligned
    # accumulation of 4- and 2-byte elements one at a time
    (S, BF16, [0], [2000001], True, "KERNEL_ROW_WALK"),
    (BF16, S, [0, 2, 1], [21, 330, 481], True, "KERNEL_ROW_WALK"),
    (S, BF16, [0], [2000001], False, "KERNEL_ROW_SMALL"),
    (S, BF16, [0], [4000000], True, "KERNEL_ROW_SMALL"),
    (S, D, [0], [2000001], True, "KERNEL_ROW"),
    (S, BF16, [0], [20001], True, "KERNEL_ROW_SMALL"),
])
def test_row_copies_that_are_walked(tA, tB, perm, size, beta, kernel):
    one, _ = launch(tA, tB, perm, size, beta)
    assert one["kernel"] == getattr(rt, kernel), one


def test_slivers_are_walked():
    walks = (rt.KERNEL_TILE_WALK, rt.KERNEL_BOX)
    assert launch(BF16, BF16, [1, 4, 3, 0, 2], [2, 540, 723, 5, 28], True)[0]["kernel"] in walks
    assert launch(BF16, BF16, [1, 0], [2, 1600001])[0]["kernel"] in walks
    assert launch(BF16, BF16, [1, 0], [2, 1600001], family=2)[0]["kernel"] == rt.KERNEL_TILE_WALK
    # slots of over 6 times the bytes, in a group of 18
    assert launch(BF16, BF16, [3, 0, 2, 1], [32, 16128, 18, 2], True, vec_a=1, vec_b=1)[0]["kernel"] in walks
    assert launch(BF16, BF16, [1, 0], [2, 400001])[0]["kernel"] == rt.KERNEL_TILE_SMALL  # few tiles
    assert launch(BF16, BF16, [1, 0], [16, 200001])[0]["kernel"] == rt.KERNEL_TILE


def test_bench_names_the_kernel():
    import bench
    name = lambda *a, **k: bench.kernel_name(rt.Plan(*a, **k))
    assert name(D, D, [1, 0], [4000, 4100], config=dict(family=2, tile=[64, 64], vec_a=1, vec_b=2)) == \
        "ttc::transpose_lane_kernel<ttc::OpDD, 1, 2, true, false, 1>"
    assert name(S, S, [1, 0], [300, 200], beta_is_zero=True, config=dict(vec_a=1, vec_b=1)) == \
        "ttc::transpose_small_kernel<ttc::OpF32<float, float>, 1, 1, false, false, 2>"
    assert name(S, S, [1, 0], [300, 200], config=dict(vec_a=1, vec_b=1, wg_per_cu=2)) == \
        "ttc::transpose_rc_kernel<ttc::OpF32<float, float>, 1, 1, true, false, false>"
    assert name(S, S, [0, 2, 1], [127, 300, 2000], beta_is_zero=True) == \
        "ttc::row_once_kernel<ttc::OpF32<float, float>, 4, 1, true>"
