"""Performance cases: the transpositions that programs have this library do.

A case is a dict of plain values.  `path` says through which entry point it
runs:

  plan    runtime.Plan.execute: a plan made once, executed on device buffers
  legacy  runtime.legacy_transpose: the synchronous drop-in of the generated
          wrappers (plans are cached per argument set by the library)
  fp8     runtime.Plan.execute_fp8: cast-transpose with amax, delayed or
          current scaling
  batch   runtime.Batch.execute: many independent transpositions per launch

Texts hold lists ("1,0,2"); `ta` / `tb` are the type names of the C ABI.  The
plan is the library's own choice (no tuning), as a program gets it that only
calls ttc_plan_create.
"""
import math

import numpy as np
import torch

from ttc_amd import runtime as rt
from ttc_amd import workloads as wl

TYPES = {"s": rt.S, "d": rt.D, "c": rt.C, "z": rt.Z, "bf16": rt.BF16, "f16": rt.F16, "e4m3": rt.E4M3,
         "e5m2": rt.E5M2}
FP8_MAX = {"e4m3": 448.0, "e5m2": 57344.0}
WIDE = {"s": torch.float64, "d": torch.float64, "bf16": torch.float64, "f16": torch.float64,
        "c": torch.complex128, "z": torch.complex128}
BATCH_TYPES = {rt.S: "s", rt.D: "d", rt.BF16: "bf16"}
DEV = "cuda:0"


def _ints(text):
    return [int(x) for x in text.split(",")] if text else None


def _text(values):
    return ",".join(str(int(v)) for v in values)


def _single(name, path, ta, tb, perm, size, alpha=1.0, beta=0.0, lda=None, ldb=None, **more):
    c = {"name": name, "path": path, "ta": ta, "tb": tb, "perm": _text(perm), "size": _text(size),
         "alpha": float(alpha), "beta": float(beta), "lda": _text(lda) if lda else "", "ldb": _text(ldb) if ldb else ""}
    c.update(more)
    return c


def listed():
    c2 = wl.plain_c2()

    def c2_case(name, k, t, beta):
        es = {"s": 4, "d": 8}[t]
        c = c2[k]
        return _single(name, "plan", t, t, c["perm"], c["sizes"][es], 1.0, beta, c["lda"] and c["lda"][es],
                       c["ldb"] and c["ldb"][es])

    c1, c3, (f2, f4) = wl.plain_c1(), wl.mixed_c3(), wl.fp8_c4()
    return [
        # the smallest calls: a 48 KiB block of a larger computation, where
        # the call and the launch are what a program waits for
        _single("tiny_s_102", "plan", "s", "s", [1, 0, 2], [32, 24, 16], 1.0, 0.0),
        # a contraction's operand brought into matrix order: fp64, rank 4,
        # ragged extents, a few hundred KiB, accumulated into B
        _single("small_d_2031", "plan", "d", "d", [2, 0, 3, 1], [37, 21, 19, 5], 1.0, 1.0),
        # sequence and head dimensions exchanged in bf16 (rows stay whole)
        _single("heads_bf16_0213", "plan", "bf16", "bf16", [0, 2, 1, 3], [128, 512, 16, 4], 1.0, 0.0),
        # a medium matrix with ragged sides through the drop-in wrapper, as
        # programs call the functions TTC generates
        _single("dropin_s_10", "legacy", "s", "s", [1, 0], [1501, 1103], 1.0, 0.0),
        # medium complex tensor, rank 3, all dimensions reversed
        _single("medium_c_210", "plan", "c", "c", [2, 1, 0], [96, 80, 110], 1.3, 0.0),
        # the benchmark configuration of the reference: fp32, alpha = beta = 1
        _single("c1_s_102", "plan", "s", "s", c1["perm"], c1["size"], c1["alpha"], c1["beta"]),
        # 200 MiB tensors, the size the reference benchmarks at: odd extents
        # and short leading dimensions in fp32, fp64 with accumulation, and
        # a sub-tensor of a padded tensor
        c2_case("large_s_rank6", 14, "s", 0.0),
        c2_case("large_d_rank5", 8, "d", 1.0),
        c2_case("padded_s", 15, "s", 0.0),
        # mixed precision: fp32 accumulators to bf16 with alpha and beta
        _single("mixed_s_bf16_3102", "plan", "s", "bf16", c3["perm"], c3["size"], c3["alpha"], c3["beta"]),
        # activations to fp8, transposed, current scaling (amax of this
        # tensor, then the cast)
        _single("fp8_bf16_e4m3", "fp8", "bf16", "e4m3", f2["perm"], f2["size"], 1.0, 0.0, mode="current"),
        # many independent transpositions of mixed rank, size and type in one
        # grouped launch
        {"name": "batch_64", "path": "batch", "ops": 64, "shapes": 5, "min_kib": 4, "max_kib": 65536},
    ]


PLAIN = ["s", "s", "s", "d", "d", "bf16", "bf16", "f16", "c", "z"]
MIXED = [("s", "bf16"), ("s", "f16"), ("bf16", "s"), ("s", "d"), ("d", "s"), ("c", "z"), ("z", "c")]
FP8 = [("s", "e4m3"), ("bf16", "e4m3"), ("f16", "e4m3"), ("bf16", "e5m2"), ("s", "e5m2")]


def _draw_extents(rng, rank, n):
    """Log-uniform proportions scaled to about n elements, every extent >= 2."""
    base = [math.exp(rng.uniform(0.0, math.log(256.0))) for _ in range(rank)]
    f = (n / math.prod(base)) ** (1.0 / rank)
    ext = [max(2, round(b * f)) for b in base]
    big = max(range(rank), key=lambda i: ext[i])
    ext[big] = max(2, n // math.prod(e for i, e in enumerate(ext) if i != big))
    return ext


def draw(rng):
    kind = rng.choice(["plan"] * 6 + ["legacy", "fp8", "fp8", "batch"])
    if kind == "batch":
        return {"path": "batch", "ops": rng.randrange(6, 65), "shapes": rng.randrange(1, 1 << 20), "min_kib": 4,
                "max_kib": int(2 ** rng.uniform(8, 14))}
    if kind == "fp8":
        ta, tb = rng.choice(FP8)
    elif rng.random() < 0.25:
        ta, tb = rng.choice(MIXED)
    else:
        ta = tb = rng.choice(PLAIN)
    wide = max(rt.DTYPE_BYTES[TYPES[ta]], rt.DTYPE_BYTES[TYPES[tb]])
    # 16 KiB to 200 MiB on the wider side
    nbytes = math.exp(rng.uniform(math.log(16 << 10), math.log(200 << 20)))
    rank = rng.randrange(2, 7)
    size = _draw_extents(rng, rank, int(nbytes / wide))
    while math.prod(size) * wide > (208 << 20):
        big = max(range(rank), key=lambda i: size[i])
        size[big] = max(2, size[big] // 2)
    # half of the shapes are ragged, half come in multiples of 8 where large enough
    if rng.random() < 0.5:
        size = [s // 8 * 8 if s >= 16 else s for s in size]
    perm = list(range(rank))
    while perm == sorted(perm):
        rng.shuffle(perm)
    lda = ldb = None
    if kind == "plan" and math.prod(size) * wide < (64 << 20) and rng.random() < 0.2:
        lda = [s + rng.randrange(0, 4) for s in size]
        ldb = [size[p] + rng.randrange(0, 4) for p in perm]
        if math.prod(lda) > 2 * math.prod(size) or math.prod(ldb) > 2 * math.prod(size):
            lda = ldb = None
    if kind == "fp8":
        c = _single("", kind, ta, tb, perm, size, rng.choice([1.0, 0.5]), 0.0, mode=rng.choice(["delayed", "current"]))
    else:
        c = _single("", kind, ta, tb, perm, size, rng.choice([1.0, 1.3]), rng.choice([0.0, 0.0, 1.0, 0.7]), lda, ldb)
    del c["name"]
    return c


def _normal(n, t, gen, scale=1.0):
    """n values of type t, normally distributed, as a flat device tensor."""
    if t in ("c", "z"):
        dt = torch.float32 if t == "c" else torch.float64
        return torch.view_as_complex((torch.randn(n, 2, generator=gen, device=DEV, dtype=dt) * scale))
    x = torch.randn(n, generator=gen, device=DEV, dtype=torch.float64 if t == "d" else torch.float32) * scale
    return x.to(rt.torch_dtype(TYPES[t]))


def _heavy(n, t, gen):
    """Activations: normal with 1% of the values ten times larger."""
    x = torch.randn(n, generator=gen, device=DEV)
    x = torch.where(torch.rand(n, generator=gen, device=DEV) < 0.01, 10.0 * x, x)
    return x.to(rt.torch_dtype(TYPES[t]))


def _generator(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    return gen


def _single_buffers(case, seed):
    perm, size = _ints(case["perm"]), _ints(case["size"])
    lda = _ints(case["lda"]) or size
    ldb = _ints(case["ldb"]) or [size[p] for p in perm]
    gen = _generator(seed)
    if case["path"] == "fp8":
        return _heavy(math.prod(lda), case["ta"], gen), torch.zeros(math.prod(ldb), dtype=torch.uint8, device=DEV)
    return _normal(math.prod(lda), case["ta"], gen), _normal(math.prod(ldb), case["tb"], gen)


def _batch_ops(case):
    """The case's ops and, per type, how many elements their buffers take
    (each op's A and B start 256-byte aligned in one buffer per type)."""
    ops = wl.batch_c5(case["ops"], case["shapes"], case["min_kib"] << 10, case["max_kib"] << 10)
    used = {t: 0 for t in BATCH_TYPES}
    for o in ops:
        o["n"] = math.prod(o["size"])
        o["at"] = used[o["type"]]
        used[o["type"]] += -(-o["n"] // 128) * 128
    return ops, used


def _batch_buffers(case, seed):
    ops, used = _batch_ops(case)
    gen = _generator(seed)
    bufs = {}
    for t, n in used.items():
        if n:
            bufs[t] = (_normal(n, BATCH_TYPES[t], gen), _normal(n, BATCH_TYPES[t], gen))
    return ops, bufs


def prepare(case, seed):
    if case["path"] == "batch":
        ops, bufs = _batch_buffers(case, seed)
        recs = []
        for o in ops:
            A, B = bufs[o["type"]]
            recs.append({"type_a": o["type"], "type_b": o["type"], "perm": o["perm"], "size": o["size"],
                         "A": A[o["at"]:o["at"] + o["n"]], "B": B[o["at"]:o["at"] + o["n"]], "alpha": o["alpha"],
                         "beta": o["beta"]})
        return {"path": "batch", "batch": rt.Batch(recs), "bufs": bufs}
    A, B = _single_buffers(case, seed)
    st = {"path": case["path"], "A": A, "B": B, "alpha": case["alpha"], "beta": case["beta"],
          "ta": TYPES[case["ta"]], "tb": TYPES[case["tb"]], "perm": _ints(case["perm"]), "size": _ints(case["size"]),
          "lda": _ints(case["lda"]), "ldb": _ints(case["ldb"])}
    if case["path"] != "legacy":
        st["plan"] = rt.Plan(st["ta"], st["tb"], st["perm"], st["size"], st["lda"], st["ldb"],
                             beta_is_zero=case["beta"] == 0.0)
    if case["path"] == "fp8":
        st["mode"] = rt.SCALE_CURRENT if case["mode"] == "current" else rt.SCALE_DELAYED
        # delayed scaling: the scale of the previous step's tensor
        st["scale"] = torch.full((1,), FP8_MAX[case["tb"]] / 50.0, device=DEV)
        st["amax"] = torch.zeros(1, device=DEV)
        st["scale_inv"] = torch.zeros(1, device=DEV)
    return st


def run(state):
    st = state
    if st["path"] == "plan":
        st["plan"].execute(st["A"], st["B"], st["alpha"], st["beta"])
        return st["B"]
    if st["path"] == "legacy":
        rt.legacy_transpose(st["ta"], st["tb"], st["A"], st["B"], st["alpha"], st["beta"], st["perm"], st["size"],
                            st["lda"], st["ldb"])
        return st["B"]
    if st["path"] == "fp8":
        st["plan"].execute_fp8(st["A"], st["B"], st["alpha"], scale_in=st["scale"], amax_out=st["amax"],
                               scale_inv_out=st["scale_inv"], mode=st["mode"])
        return {"B": st["B"], "amax": st["amax"], "scale_inv": st["scale_inv"]}
    st["batch"].execute()
    return {BATCH_TYPES[t]: b for t, (_, b) in st["bufs"].items()}


def work(case):
    if case["path"] == "batch":
        nbytes = sum(wl.algorithmic_bytes(o["n"], rt.DTYPE_BYTES[o["type"]], rt.DTYPE_BYTES[o["type"]],
                                          o["beta"] == 0) for o in _batch_ops(case)[0])
        return {"bytes": nbytes, "flops": 0}
    n = math.prod(_ints(case["size"]))
    return {"bytes": wl.algorithmic_bytes(n, rt.DTYPE_BYTES[TYPES[case["ta"]]], rt.DTYPE_BYTES[TYPES[case["tb"]]],
                                          case["beta"] == 0.0), "flops": 0}


def _exact_single(A, B, ta, tb, perm, size, lda, ldb, alpha, beta):
    """B after B[perm(i)] = alpha A[i] + beta B[perm(i)] in 64 bits (index 0
    is the fastest, so the torch views have their dimensions reversed)."""
    r = len(size)
    lda, ldb = lda or size, ldb or [size[p] for p in perm]
    a = A.to(WIDE[ta]).reshape(lda[::-1])[tuple(slice(0, s) for s in size[::-1])]
    out = B.to(WIDE[tb]).clone()
    b = out.view(ldb[::-1])[tuple(slice(0, size[p]) for p in perm[::-1])]
    a = a.permute([r - 1 - p for p in perm[::-1]])
    b.copy_(alpha * a + beta * b if beta != 0.0 else alpha * a)
    return out


def exact(case, seed):
    if case["path"] == "batch":
        ops, bufs = _batch_buffers(case, seed)
        outs = {t: b.to(torch.float64) for t, (_, b) in bufs.items()}
        for o in ops:
            A, B = bufs[o["type"]]
            t = BATCH_TYPES[o["type"]]
            s = slice(o["at"], o["at"] + o["n"])
            outs[o["type"]][s] = _exact_single(A[s], B[s], t, t, o["perm"], o["size"], None, None, o["alpha"],
                                               o["beta"])
        return {BATCH_TYPES[t]: x for t, x in outs.items()}
    A, B = _single_buffers(case, seed)
    if case["path"] == "fp8":
        amax = (A.to(torch.float64) * case["alpha"]).abs().max().reshape(1)
        top = FP8_MAX[case["tb"]]
        inv = amax / top if case["mode"] == "current" else torch.full_like(amax, 1.0 / float(np.float32(top / 50.0)))
        return {"B": None, "amax": amax, "scale_inv": inv}
    return _exact_single(A, B, case["ta"], case["tb"], _ints(case["perm"]), _ints(case["size"]), _ints(case["lda"]),
                         _ints(case["ldb"]), case["alpha"], case["beta"])
