"""GPU parity of row copies in grouped launches, bit-exact against the oracle:
by row length (every vector width, aligned and unaligned, beta read or not,
dense, padded and misaligned, all in one launch per type), and ops whose
configuration names a tile."""
import pytest

from common import CODE, first_diff, from_device, make_case, oracle_run, same_bits, to_device

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 15, 16, 17, 24, 31, 32, 33, 64, 127, 128, 129]


@pytest.mark.parametrize("code", ["s", "d", "c", "z", "b", "h"])
def test_row_lengths_in_one_launch(gpu, code):
    import torch
    from ttc_amd import runtime as rt
    t, _ = CODE[code]
    ops, kinds = [], set()
    for n0 in ROWS:
        for pad in (0, 1):
            size = [n0, 13, 22]
            lda = [n0 + 3, 13, 23] if pad else None
            ldb = [n0 + 1, 24, 13] if pad else None
            for beta in (0.0, 0.75):
                for off in (0, 1):
                    A, B = make_case(t, t, [0, 2, 1], size, lda, ldb, seed=n0 + pad)
                    dA = torch.zeros(A.nbytes + 16, dtype=torch.uint8, device=gpu)
                    dB = torch.zeros(B.nbytes + 16, dtype=torch.uint8, device=gpu)
                    o = off * A.itemsize
                    dA[o:o + A.nbytes], dB[o:o + B.nbytes] = to_device(A, gpu), to_device(B, gpu)
                    launch = rt.Plan(t, t, [0, 2, 1], size, lda, ldb, beta == 0.0).launch()
                    kinds.add((launch["vec_a"], launch["unaligned"], beta))
                    ops.append(dict(type_a=t, perm=[0, 2, 1], size=size, lda=lda, ldb=ldb, alpha=1.25, beta=beta,
                                    A=dA[o:o + A.nbytes], B=dB[o:o + B.nbytes], n0=n0, hB=B,
                                    want=oracle_run(t, t, A, B, 1.25, beta, [0, 2, 1], size, lda, ldb)))
    assert len(kinds) >= {"s": 6, "d": 4, "c": 4, "z": 2, "b": 9, "h": 9}[code], kinds
    batch = rt.Batch(ops)
    batch.execute()
    torch.cuda.synchronize()
    for o in ops:
        got = from_device(o["B"], o["hB"])
        assert same_bits(got, o["want"]), (code, o["n0"], o["beta"], o["lda"], first_diff(got, o["want"]))


@pytest.mark.parametrize("code,n0", [("s", 54), ("s", 8), ("d", 6), ("b", 4), ("b", 48), ("h", 100), ("c", 6)])
@pytest.mark.parametrize("beta", [0.0, 0.75])
def test_tiles_on_whole_rows(gpu, code, n0, beta):
    """A box tile of an op that keeps dimension 0 in place, at widths that
    grouped box tiles do not have: the op runs without its tile."""
    import torch
    from ttc_amd import runtime as rt
    t, _ = CODE[code]
    ops = []
    for size, perm, tile in (([n0, 13, 22], [0, 2, 1], [n0, 4, 2]), ([n0], [0], [n0])):
        for vec_b in (0, 1):
            A, B = make_case(t, t, perm, size, seed=n0)
            ops.append(dict(type_a=t, perm=perm, size=size, alpha=1.25, beta=beta, A=to_device(A, gpu),
                            B=to_device(B, gpu), config=dict(tile=tile, vec_b=vec_b), hB=B,
                            want=oracle_run(t, t, A, B, 1.25, beta, perm, size)))
    batch = rt.Batch(ops)
    batch.execute()
    torch.cuda.synchronize()
    for o in ops:
        got = from_device(o["B"], o["hB"])
        assert same_bits(got, o["want"]), (code, o["size"], o["config"], first_diff(got, o["want"]))
