"""GPU parity of row x column launches whose work-groups walk several tiles,
which a plan takes for wg_per_cu and for an explicit tile with lds_buffers:
every type pair, both buffer counts, all tile orders (padding ids of grouped
orders included), padded tensors, A offsets past 2^30, and casts to fp8; each
case first asserts that this kernel is the one launched."""
import numpy as np
import pytest

from common import (BF16, CODE, F16, S, _real_update, first_diff, from_device, make_case, oracle_run, same_bits,
                    to_device)
from oracle import oracle as orc
from test_gpu_cast_batch import E4M3, E5M2, FP8_MAX, _heavy_input
from test_gpu_parity import RANDOM_SHAPES, check

pytestmark = pytest.mark.gpu


def walks(tA, tB, perm, size, lda=None, ldb=None, bz=True, **cfg):
    from ttc_amd import runtime as rt
    launch = rt.Plan(tA, tB, perm, size, lda, ldb, bz, cfg).launch()
    assert launch["kernel"] == rt.KERNEL_TILE_WALK, (launch, cfg)
    return launch


@pytest.mark.parametrize("code", ["s", "d", "c", "z", "sd", "ds", "cz", "zc", "b", "h", "sb", "sh", "bs", "hs"])
def test_random_shapes(gpu, code):
    from ttc_amd import runtime as rt
    tA, tB = CODE[code]
    n = 0
    for i, (perm, size) in enumerate(RANDOM_SHAPES):
        if perm[0] == 0 or rt.fuse_indices(perm, size, None, None)[0] == [0]:
            continue
        for j, beta in enumerate((0.0, 0.7)):
            cfg = dict(family=2, wg_per_cu=1 + (i + j) % 3, tile_order=1 + (i + 2 * j) % 4,
                       lds_buffers=1 + (i + j) % 2, grid_order=(i + j) % 5)
            lda = [s + 1 + k % 3 for k, s in enumerate(size)] if i % 3 == 0 else None
            ldb = [size[p] + 2 for p in perm] if i % 4 == 0 else None
            launch = walks(tA, tB, perm, size, lda, ldb, beta == 0, **cfg)
            assert launch["lds_buffers"] == cfg["lds_buffers"]
            check(gpu, tA, tB, perm, size, 1.3, beta, lda, ldb, seed=100 + i, dist="outliers", config=cfg)
            n += 1
    assert n >= 16


def test_grouped_tile_orders_with_padding_ids(gpu):
    """65 tiles along the rows in groups of 8 / 16 leave padding ids, which the
    walk processes (B read and written) as empty tiles."""
    for order, ids in ((3, 2376), (4, 2640)):
        for buffers in (1, 2):
            for beta in (0.0, 0.75):
                cfg = dict(family=2, tile=[62, 128], vec_a=2, vec_b=2, tile_order=order, lds_buffers=buffers)
                launch = walks(BF16, BF16, [1, 0], [4000, 4100], bz=beta == 0, **cfg)
                assert launch["units"] == ids and launch["lane_fixed"] == 1
                check(gpu, BF16, BF16, [1, 0], [4000, 4100], 1.5, beta, seed=order, config=cfg)


def test_padded_leading_dimensions_on_lane_fixed_tiles(gpu):
    for i, (tA, tB, size, tile) in enumerate(((BF16, BF16, [4000, 4100], [62, 128]), (S, BF16, [2048, 8200], [128, 64]),
                                              (BF16, S, [1920, 9000], [124, 62]))):
        lda, ldb = [s + 3 for s in size], [s + 5 for s in size[::-1]]
        for buffers in (1, 2):
            cfg = dict(family=2, tile=tile, vec_a=1, vec_b=1, lds_buffers=buffers)
            assert walks(tA, tB, [1, 0], size, lda, ldb, False, **cfg)["lane_fixed"] == 1
            check(gpu, tA, tB, [1, 0], size, 0.5, 1.0, lda, ldb, seed=i, config=cfg)


def test_a_offsets_past_2_30(gpu):
    """fp32 -> bf16 on [128, 1, 1, 64] tiles that span 1.6 GB of A; sampled
    outputs bit for bit."""
    import torch
    from test_gpu_workloads import C3_PERM, C3_SIZE, NSAMPLE, _draw, _offsets
    from ttc_amd import runtime as rt
    cfg = {"family": 2, "tile": [128, 1, 1, 64], "lds_buffers": 2}
    assert walks(S, BF16, C3_PERM, C3_SIZE, bz=False, **cfg)["lane_fixed"] == 1
    n = int(np.prod(C3_SIZE))
    gen = torch.Generator(device=gpu)
    gen.manual_seed(32)
    A = _draw(torch, n, gpu, gen, torch.float32)
    B = _draw(torch, n, gpu, gen, torch.bfloat16)
    offA, offB = _offsets(C3_PERM, C3_SIZE, np.random.default_rng(35), NSAMPLE)
    tiA, tiB = torch.from_numpy(offA).to(gpu), torch.from_numpy(offB).to(gpu)
    a, b = A[tiA].cpu(), B[tiB].cpu()
    rt.Plan(S, BF16, C3_PERM, C3_SIZE, beta_is_zero=False, config=cfg).execute(A, B, 1.3, 0.7)
    torch.cuda.synchronize()
    want = _real_update(S, BF16, a.numpy(), b.view(torch.int16).numpy().view(np.uint16), 1.3, 0.7, False)
    assert np.array_equal(B[tiB].cpu().view(torch.int16).numpy().view(np.uint16), want)


@pytest.mark.parametrize("tA,tB", [(S, E4M3), (BF16, E4M3), (F16, E5M2)])
def test_fp8_casts(gpu, tA, tB):
    import torch
    from ttc_amd import runtime as rt
    cases = [([1, 0], [1031, 2050], dict(tile=[64, 32], vec_a=1, vec_b=1, lds_buffers=2)),
             ([1, 0], [4096, 2100], dict(tile=[64, 62], vec_a=2, vec_b=1, lds_buffers=1, tile_order=3)),
             ([2, 0, 1], [33, 17, 400], dict(wg_per_cu=2)), ([1, 0], [512, 448], dict(wg_per_cu=1, lds_buffers=1))]
    for i, (perm, size, cfg) in enumerate(cases):
        walks(tA, tB, perm, size, family=2, **cfg)
        plan = rt.Plan(tA, tB, perm, size, beta_is_zero=True, config=dict(family=2, **cfg))
        n = int(np.prod(size))
        A = _heavy_input(tA, n, 60 + i)
        dA, dB = to_device(A, gpu), torch.zeros(n, dtype=torch.uint8, device=gpu)
        amax = torch.full((1,), -1.0, dtype=torch.float32, device=gpu)
        want = np.zeros(n, np.uint8)
        top = orc.cast_fp8(tA, tB, A, want, 0.5, 3.5, perm, size)
        plan.execute_fp8(dA, dB, 0.5, scale=3.5, amax_out=amax)
        torch.cuda.synchronize()
        got = dB.cpu().numpy()
        assert same_bits(got, want) and float(amax.item()) == top, (tA, tB, size, first_diff(got, want))
        scale = np.float32(FP8_MAX[tB]) / np.float32(top)
        orc.cast_fp8(tA, tB, A, want, 0.5, float(scale), perm, size)
        plan.execute_fp8(dA, dB, 0.5, amax_out=amax, mode=rt.SCALE_CURRENT)
        torch.cuda.synchronize()
        assert same_bits(dB.cpu().numpy(), want) and float(amax.item()) == top, (tA, tB, size, "current")


@pytest.mark.parametrize("code", ["s", "d", "b", "c", "sb"])
@pytest.mark.parametrize("perm,size", [([1, 0], [2, 1600001]), ([1, 0], [1600001, 3]), ([1, 2, 0], [3, 249, 7000])])
def test_slivers(gpu, code, perm, size):
    """Short groups, whose tiles are walked where one work-group per tile would
    leave slivers."""
    import torch
    from ttc_amd import runtime as rt
    tA, tB = CODE[code]
    for beta in (0.0, 0.75):
        A, B = make_case(tA, tB, perm, size, seed=len(size))
        dA, dB = to_device(A, gpu), to_device(B, gpu)
        plan = rt.Plan(tA, tB, perm, size, beta_is_zero=beta == 0.0)
        plan.execute(dA, dB, 1.25, beta)
        torch.cuda.synchronize()
        got, want = from_device(dB, B), oracle_run(tA, tB, A, B, 1.25, beta, perm, size)
        assert same_bits(got, want), (plan.launch(), first_diff(got, want))


@pytest.mark.parametrize("code", ["s", "d", "b", "h", "c", "sb", "bs"])
@pytest.mark.parametrize("perm,size", [([1, 5, 0, 2, 4, 3], [6, 6, 14, 14, 46, 6]), ([1, 0, 2], [512, 64, 40]),
                                       ([1, 0], [1024, 6]), ([3, 1, 2, 4, 5, 0], [24, 3, 24, 2, 2, 40])])
def test_misaligned_pointers_take_a_tile_of_their_own(gpu, code, perm, size):
    import torch
    from ttc_amd import runtime as rt
    tA, tB = CODE[code]
    for beta in (0.0, 0.75):
        A, B = make_case(tA, tB, perm, size, seed=len(size))
        dA = torch.zeros(A.nbytes + 16, dtype=torch.uint8, device=gpu)
        dB = torch.zeros(B.nbytes + 16, dtype=torch.uint8, device=gpu)
        a, b = dA[A.itemsize:A.itemsize + A.nbytes], dB[B.itemsize:B.itemsize + B.nbytes]
        a.copy_(to_device(A, gpu))
        b.copy_(to_device(B, gpu))
        plan = rt.Plan(tA, tB, perm, size, beta_is_zero=beta == 0.0)
        plan.execute(a, b, 1.25, beta)
        torch.cuda.synchronize()
        got, want = from_device(b, B), oracle_run(tA, tB, A, B, 1.25, beta, perm, size)
        assert same_bits(got, want), (plan.launch(), first_diff(got, want))
        assert not dB[:B.itemsize].any() and not dB[B.itemsize + B.nbytes:].any()
