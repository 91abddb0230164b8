"""Kernel-instance generator for libttc_hip.so.

Writes ttc_amd/csrc/gen/inst_<pair>.hip, one file per (A type, B type) pair,
each listing the template instances of the hand-written kernels
(csrc/ttc_kernels.hpp box tiles, csrc/ttc_rc.hpp row x column tiles,
csrc/ttc_row.hpp row copy) for every vector width and store mode, plus
gen/inst_all.h, the table the runtime searches.  This plays the role of
TTC's per-transposition code generation (ttc/GPUtransposeGenerator.py:
720-758, ttc/CUDAtranspose.py:114-176): instead of emitting one kernel per
(perm, size) and compiling it per request, the shape becomes kernel
arguments and the generator emits the finite set of type/vector/mode
variants once, at build time.
"""
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
GEN_DIR = os.path.join(_HERE, "csrc", "gen")

# (ttc_dtype_t name, C++ storage type, bytes)
TYPES = {
    "S": ("float", 4), "D": ("double", 8), "C": ("c32", 8), "Z": ("c64", 16),
    "BF16": ("bf16s", 2), "F16": ("f16s", 2), "E4M3": ("e4m3s", 1), "E5M2": ("e5m2s", 1),
}

F32_CLASS = ("S", "BF16", "F16")


def vec_widths(nbytes):
    """Same rule as ttc::vec_widths (csrc/ttc_plan.h)."""
    w = [1]
    if nbytes <= 8:
        w.append(2)
    wide = 16 // nbytes
    if wide > 2:
        w.append(wide)
    return w


def row_widths(na, nb):
    """Same rule as ttc::row_widths (csrc/ttc_plan.h): vector widths of the
    row-copy kernel, one width for both sides, at most 16 bytes on each."""
    w = [1]
    wide = 16 // max(na, nb)
    if wide >= 2:
        w.append(2)
    if wide > 2:
        w.append(wide)
    return w


def row_unaligned_widths(na, nb):
    """The widths ttc::row_unaligned_width (csrc/ttc_plan.h) may return beside 1:
    vectors of the row copy in unaligned vectors."""
    w = []
    v = 2
    while v * max(na, nb) <= 16:
        w.append(v)
        v *= 2
    return w


def row_unaligned_modes(na, nb, modes):
    """Store modes it is instantiated for (csrc/ttc_plan.h
    row_unaligned_mode)."""
    return [m for m in modes if m in ("kModeBz", "kModeFp8") or (m == "kModeBeta" and max(na, nb) <= 2)]


def op_for(ta, tb):
    if ta in F32_CLASS and tb in F32_CLASS:
        return "OpF32<%s, %s>" % (TYPES[ta][0], TYPES[tb][0])
    if tb in ("E4M3", "E5M2") and ta in F32_CLASS:
        return "OpF8<%s, %s>" % (TYPES[ta][0], TYPES[tb][0])
    return {("D", "D"): "OpDD", ("S", "D"): "OpSD", ("D", "S"): "OpDS", ("C", "C"): "OpCC",
            ("Z", "Z"): "OpZZ", ("C", "Z"): "OpCZ", ("Z", "C"): "OpZC"}[(ta, tb)]


def pairs():
    out = []
    for ta in F32_CLASS:
        for tb in F32_CLASS:
            if {ta, tb} != {"BF16", "F16"}:
                out.append((ta, tb))
    out += [("D", "D"), ("S", "D"), ("D", "S"), ("C", "C"), ("Z", "Z"), ("C", "Z"), ("Z", "C")]
    for ta in F32_CLASS:
        for tb in ("E4M3", "E5M2"):
            out.append((ta, tb))
    return out


def instance_files(ta, tb):
    """One file per (pair, A vector width), so the build parallelises."""
    op = op_for(ta, tb)
    fp8 = tb in ("E4M3", "E5M2")
    modes = ["kModeFp8"] if fp8 else ["kModeBeta", "kModeBz", "kModeBzNt"]
    out = []
    for va in vec_widths(TYPES[ta][1]):
        lines = []
        for vb in vec_widths(TYPES[tb][1]):
            for m in modes:
                lines.append("      make_entry<%s, %d, %d, %s>(TTC_%s, TTC_%s)," % (op, va, vb, m, ta, tb))
                # row x column tile family
                lines.append("      make_rc_entry<%s, %d, %d, %s>(TTC_%s, TTC_%s)," % (op, va, vb, m, ta, tb))
        name = "inst_%s_%s_va%d" % (ta.lower(), tb.lower(), va)
        src = []
        src.append("// Generated by ttc_amd/gen_instances.py -- do not edit.")
        src.append('#include "../ttc_launch.hpp"')
        src.append("namespace ttc {")
        src.append("const KernelEntry* %s(int* n) {" % name)
        src.append("  static const KernelEntry entries[] = {")
        src += lines
        src.append("  };")
        src.append("  *n = (int)(sizeof(entries) / sizeof(entries[0]));")
        src.append("  return entries;")
        src.append("}")
        src.append("}  // namespace ttc")
        out.append((name, "\n".join(src) + "\n", len(lines)))
    # row-copy family (perm[0] == 0), one file per pair
    lines = ["      make_row_entry<%s, %d, %s>(TTC_%s, TTC_%s)," % (op, v, m, ta, tb)
             for v in row_widths(TYPES[ta][1], TYPES[tb][1]) for m in modes]
    lines += ["      make_row_unaligned_entry<%s, %d, %s>(TTC_%s, TTC_%s)," % (op, v, m, ta, tb)
              for v in row_unaligned_widths(TYPES[ta][1], TYPES[tb][1])
              for m in row_unaligned_modes(TYPES[ta][1], TYPES[tb][1], modes)]
    name = "inst_%s_%s_row" % (ta.lower(), tb.lower())
    src = ["// Generated by ttc_amd/gen_instances.py -- do not edit.", '#include "../ttc_launch.hpp"',
           "namespace ttc {", "const KernelEntry* %s(int* n) {" % name, "  static const KernelEntry entries[] = {"]
    src += lines
    src += ["  };", "  *n = (int)(sizeof(entries) / sizeof(entries[0]));", "  return entries;", "}",
            "}  // namespace ttc"]
    out.append((name, "\n".join(src) + "\n", len(lines)))
    return out


def generate(out_dir=GEN_DIR):
    os.makedirs(out_dir, exist_ok=True)
    names = []
    total = 0
    for ta, tb in pairs():
        for name, text, n in instance_files(ta, tb):
            total += n
            path = os.path.join(out_dir, name + ".hip")
            if not os.path.exists(path) or open(path).read() != text:
                with open(path, "w") as f:
                    f.write(text)
            names.append(name)
    keep = set(n + ".hip" for n in names) | {"inst_all.h"}
    for f in os.listdir(out_dir):
        if f not in keep:
            os.remove(os.path.join(out_dir, f))
    hdr = ["// Generated by ttc_amd/gen_instances.py -- do not edit.", "#pragma once",
           '#include "../ttc_launch.hpp"', "namespace ttc {"]
    for n in names:
        hdr.append("const KernelEntry* %s(int* n);" % n)
    hdr.append("typedef const KernelEntry* (*InstanceList)(int*);")
    hdr.append("static const InstanceList kInstanceLists[] = {")
    for n in names:
        hdr.append("    &%s," % n)
    hdr.append("};")
    hdr.append("}  // namespace ttc")
    text = "\n".join(hdr) + "\n"
    path = os.path.join(out_dir, "inst_all.h")
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as f:
            f.write(text)
    return [os.path.join(out_dir, n + ".hip") for n in names], total


if __name__ == "__main__":
    files, total = generate()
    print("%d instance files, %d kernels" % (len(files), total))
