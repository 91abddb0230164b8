"""GPU parity of casts to fp8 that keep amax over more than 256 tiles or
chunks, where most work-groups take two: odd counts, partial tiles, unaligned
and short rows, delayed and current scaling (whose cast walks backwards), and
the largest element at many places; B and amax bit for bit."""
import numpy as np
import pytest

from common import BF16, F16, S, first_diff, same_bits, to_device
from oracle import oracle as orc
from test_gpu_cast_batch import E4M3, E5M2, FP8_MAX, _heavy_input

pytestmark = pytest.mark.gpu

SHAPES = [  # perm, size
    ([1, 0], [1024, 4096]), ([1, 0], [1031, 2050]), ([1, 0], [2049, 515]), ([2, 0, 1], [130, 33, 257]),
    ([0, 2, 1], [127, 300, 121]), ([0, 2, 1], [128, 150, 250]), ([0, 2, 1], [9, 700, 450]),
    ([0, 2, 1], [5, 1000, 333]), ([0, 2, 1], [127, 200, 121]),
]


@pytest.mark.parametrize("tA,tB", [(S, E4M3), (S, E5M2), (BF16, E4M3), (F16, E5M2)])
@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_amax_over_many_units(gpu, tA, tB, case):
    from ttc_amd import runtime as rt
    perm, size = SHAPES[case]
    launch = rt.Plan(tA, tB, perm, size, beta_is_zero=True).launch()
    # (rows on aligned vectors are walked at these sizes, and so are 257 to 512 chunks with amax)
    rows = rt.KERNEL_ROW if launch["unaligned"] else rt.KERNEL_ROW_WALK
    assert launch["units"] > 256 and launch["kernel"] == (rows if perm[0] == 0 else rt.KERNEL_TILE), launch
    run_case(gpu, tA, tB, perm, size, 70 + case)


def test_amax_over_many_aligned_chunks(gpu):
    from ttc_amd import runtime as rt
    launch = rt.Plan(BF16, E4M3, [0, 2, 1], [128, 4096, 256], beta_is_zero=True).launch()
    assert launch["units"] > 10000 and launch["kernel"] == rt.KERNEL_ROW and not launch["unaligned"], launch
    run_case(gpu, BF16, E4M3, [0, 2, 1], [128, 4096, 256], 90)


def run_case(gpu, tA, tB, perm, size, seed):
    import torch
    from ttc_amd import runtime as rt
    plan = rt.Plan(tA, tB, perm, size, beta_is_zero=True)
    launch = plan.launch()
    n = int(np.prod(size))
    A = _heavy_input(tA, n, seed)
    want = np.zeros(n, np.uint8)
    top = orc.cast_fp8(tA, tB, A, want, 0.5, 3.5, perm, size)
    dA, dB = to_device(A, gpu), torch.zeros(n, dtype=torch.uint8, device=gpu)
    amax = torch.full((1,), -1.0, dtype=torch.float32, device=gpu)
    plan.execute_fp8(dA, dB, 0.5, scale=3.5, amax_out=amax)
    torch.cuda.synchronize()
    got = dB.cpu().numpy()
    assert same_bits(got, want) and float(amax.item()) == top, (launch, first_diff(got, want))
    scale = np.float32(FP8_MAX[tB]) / np.float32(top)
    orc.cast_fp8(tA, tB, A, want, 0.5, float(scale), perm, size)
    dB.zero_()
    plan.execute_fp8(dA, dB, 0.5, amax_out=amax, mode=rt.SCALE_CURRENT)
    torch.cuda.synchronize()
    got = dB.cpu().numpy()
    assert same_bits(got, want) and float(amax.item()) == top, ("current", launch, first_diff(got, want))
    # the largest element at 40 places, those of the first and last units among them
    dt = torch.float32 if tA == S else (torch.bfloat16 if tA == BF16 else torch.float16)
    X = dA.view(dt)
    out = torch.zeros(40, device=gpu)
    places = [int(p) for p in np.linspace(0, n - 1, 40)]
    big = 32768.0
    for k, at in enumerate(places):
        old = X[at].clone()
        X[at] = -big
        plan.execute_fp8(dA, dB, 0.5, scale=1.0, amax_out=out[k:k + 1])
        X[at] = old
    torch.cuda.synchronize()
    assert top < big / 2 and out.cpu().tolist() == [big / 2] * 40
