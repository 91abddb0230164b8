"""Builds libttc_hip.so in-tree (ttc_amd/lib/) for gfx950.

  python -m ttc_amd.build [--force] [-j N]
  python -m ttc_amd.build install --prefix DIR   (library, header, pkg-config and CMake files)

Steps: write the kernel-instance files (gen_instances.py), compile every
HIP source with hipcc for gfx950 and the planner with g++, link one shared
library.  Device code is compiled with -ffp-contract=off (no FMA
contraction, as the reference's CPU oracle) and with packed-fp32
instructions disabled.
"""
import argparse
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

from . import gen_instances

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIBDIR = os.path.join(PKG, "lib")
LIB = os.path.join(LIBDIR, "libttc_hip.so")
INCLUDE = os.path.join(ROOT, "include")

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
HIP_FLAGS = [
    "-O3", "--offload-arch=" + ARCH, "-fPIC", "-std=c++17",
    "-ffp-contract=off", "-fno-gpu-flush-denormals-to-zero",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + INCLUDE, "-I" + CSRC, "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]
CXX_FLAGS = ["-O2", "-fPIC", "-std=c++17", "-Wall", "-I" + INCLUDE, "-I" + CSRC]

HEADERS = ["ttc_kernels.hpp", "ttc_rc.hpp", "ttc_lane.hpp", "ttc_row.hpp", "ttc_launch.hpp", "ttc_batch_kernels.hpp", "ttc_batch_one.hpp", "ttc_params.h",
           "ttc_plan.h", "ttc_runtime.h", "gen/inst_all.h"]
VERSION = "0.2.0"


def source_digest():
    """sha256 (first 16 hex digits) over the library's hand-written sources,
    the instance generator and the C header: what the built library reports
    in ttc_version(), so a check can tell a stale build from the checkout."""
    import hashlib
    files = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC)
                   if f.endswith((".hip", ".hpp", ".h", ".cpp")))
    files += [os.path.join(PKG, "gen_instances.py"), os.path.join(INCLUDE, "ttc_hip.h")]
    h = hashlib.sha256()
    for f in files:
        h.update(os.path.basename(f).encode() + b"\0")
        with open(f, "rb") as fh:
            h.update(fh.read())
    return h.hexdigest()[:16]


def version_string():
    return "ttc-mi355x %s (gfx950) src:%s" % (VERSION, source_digest())


def _write_version():
    """gen/ttc_version.cpp: ttc_version() of this source state (rewritten
    only when it changes, so an unchanged tree rebuilds nothing)."""
    path = os.path.join(CSRC, "gen", "ttc_version.cpp")
    text = ('// Generated by ttc_amd/build.py: the library version and a digest of its sources.\n'
            'extern "C" const char* ttc_version(void) { return "%s"; }\n' % version_string())
    os.makedirs(os.path.dirname(path), exist_ok=True)
    old = open(path).read() if os.path.exists(path) else None
    if old != text:
        with open(path, "w") as f:
            f.write(text)
    return path


def _sources():
    inst, _ = gen_instances.generate()
    batch = [os.path.join(CSRC, "ttc_batch_k_%s.hip" % pair) for pair in ("one", "s", "d", "bf16", "f16", "c", "z")]
    hip = [os.path.join(CSRC, "ttc_runtime.hip"), os.path.join(CSRC, "ttc_batch.hip")] + batch + inst
    cxx = [os.path.join(CSRC, "ttc_plan.cpp"), _write_version()]
    return hip, cxx


def _newer(src, obj, deps):
    if not os.path.exists(obj):
        return True
    t = os.path.getmtime(obj)
    return any(os.path.getmtime(d) > t for d in [src] + deps)


def _compile(cmd):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    return cmd, p.returncode, p.stdout


def build(force=False, jobs=None, verbose=False):
    """Compile and link; returns the library path.  Raises on failure."""
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    hip, cxx = _sources()
    deps = [os.path.join(CSRC, h) for h in HEADERS] + [os.path.join(INCLUDE, "ttc_hip.h")]
    cmds, objs = [], []
    for src in hip + cxx:
        obj = os.path.join(BUILD, os.path.basename(src) + ".o")
        objs.append(obj)
        if force or _newer(src, obj, deps):
            if src.endswith(".cpp"):
                cmds.append(["g++"] + CXX_FLAGS + ["-c", src, "-o", obj])
            else:
                cmds.append([HIPCC] + HIP_FLAGS + ["-x", "hip", "-c", src, "-o", obj])
    jobs = jobs or min(16, os.cpu_count() or 4)
    failed = []
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        for cmd, rc, out in ex.map(_compile, cmds):
            if verbose or rc != 0:
                sys.stderr.write(" ".join(cmd) + "\n" + out)
            if rc != 0:
                failed.append(cmd[-1])
    if failed:
        raise RuntimeError("compilation failed: %s" % ", ".join(failed))
    if force or cmds or not os.path.exists(LIB):
        tmp = LIB + ".tmp"
        link = [HIPCC, "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", tmp] + objs
        p = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        if p.returncode != 0:
            sys.stderr.write(" ".join(link) + "\n" + p.stdout)
            raise RuntimeError("link failed")
        os.replace(tmp, LIB)
    return LIB


def compile_artefacts(hip_files, out_so, libdir=LIBDIR, include=INCLUDE, rpath=None):
    """Builds emitted drop-in artefacts (<name>.hip, ttc_amd.generator) into
    one shared library linked against libttc_hip.so, as a user of the
    reference builds its generated .cu files with the rest of a program
    (ttc/Makefile:53-58): hipcc for gfx950, then -lttc_hip."""
    objs = []
    for src in hip_files:
        obj = os.path.join(BUILD, "artefact_" + os.path.basename(src) + ".o")
        os.makedirs(BUILD, exist_ok=True)
        cmd = [HIPCC, "-O2", "-fPIC", "--offload-arch=" + ARCH, "-I" + include, "-I" + os.path.dirname(src),
               "-x", "hip", "-c", src, "-o", obj]
        cmd, rc, out = _compile(cmd)
        if rc != 0:
            raise RuntimeError("artefact compilation failed: %s\n%s" % (" ".join(cmd), out))
        objs.append(obj)
    link = [HIPCC, "-shared", "-fPIC", "-o", out_so] + objs + ["-L" + libdir, "-lttc_hip",
                                                                "-Wl,-rpath," + (rpath or libdir)]
    cmd, rc, out = _compile(link)
    if rc != 0:
        raise RuntimeError("artefact link failed: %s\n%s" % (" ".join(cmd), out))
    return out_so


def pkgconfig_text(prefix, libdir, includedir):
    """pkg-config metadata of the C library (ttc_hip.pc)."""
    return "\n".join([
        "prefix=%s" % prefix, "libdir=%s" % libdir, "includedir=%s" % includedir, "",
        "Name: ttc_hip",
        "Description: Tensor transpositions for AMD Instinct MI355X (gfx950): C ABI of libttc_hip.so",
        "Version: %s" % VERSION,
        "Cflags: -I${includedir} -D__HIP_PLATFORM_AMD__ -I/opt/rocm/include",
        "Libs: -L${libdir} -Wl,-rpath,${libdir} -lttc_hip -L/opt/rocm/lib -lamdhip64", ""])


def cmake_config_text():
    """CMake package configuration: find_package(ttc_hip CONFIG) defines the
    imported target ttc::ttc_hip (library and include directory)."""
    return "\n".join([
        "# ttc_hip CMake package configuration (installed by `python -m ttc_amd.build install`).",
        "get_filename_component(_ttc_prefix \"${CMAKE_CURRENT_LIST_DIR}/../../..\" ABSOLUTE)",
        "set(ttc_hip_VERSION %s)" % VERSION,
        "set(ttc_hip_INCLUDE_DIRS \"${_ttc_prefix}/include\")",
        "set(ttc_hip_LIBRARIES \"${_ttc_prefix}/lib/libttc_hip.so\")",
        "if(NOT TARGET ttc::ttc_hip)",
        "  add_library(ttc::ttc_hip SHARED IMPORTED)",
        "  set_target_properties(ttc::ttc_hip PROPERTIES",
        "    IMPORTED_LOCATION \"${_ttc_prefix}/lib/libttc_hip.so\"",
        "    INTERFACE_INCLUDE_DIRECTORIES \"${_ttc_prefix}/include\")",
        "endif()", ""])


def install(prefix, lib=LIB):
    """Installs the C library for use without Python: <prefix>/lib/libttc_hip.so,
    <prefix>/include/ttc_hip.h, <prefix>/lib/pkgconfig/ttc_hip.pc and
    <prefix>/lib/cmake/ttc_hip/ttc_hip-config.cmake.  Emitted artefacts
    (<name>.hip / <name>.h) then build with the .pc's Cflags and Libs."""
    prefix = os.path.abspath(prefix)
    if not os.path.exists(lib):
        raise RuntimeError("libttc_hip.so is not built; run `python -m ttc_amd.build` first")
    for d in ("lib", "include", os.path.join("lib", "pkgconfig"), os.path.join("lib", "cmake", "ttc_hip")):
        os.makedirs(os.path.join(prefix, d), exist_ok=True)
    shutil.copy2(lib, os.path.join(prefix, "lib", "libttc_hip.so"))
    shutil.copy2(os.path.join(INCLUDE, "ttc_hip.h"), os.path.join(prefix, "include", "ttc_hip.h"))
    with open(os.path.join(prefix, "lib", "pkgconfig", "ttc_hip.pc"), "w") as f:
        f.write(pkgconfig_text(prefix, "${prefix}/lib", "${prefix}/include"))
    with open(os.path.join(prefix, "lib", "cmake", "ttc_hip", "ttc_hip-config.cmake"), "w") as f:
        f.write(cmake_config_text())
    return prefix


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("command", nargs="?", default="build", choices=["build", "install"])
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--prefix", default=None, help="install: destination prefix")
    ap.add_argument("-j", type=int, default=None)
    ap.add_argument("-v", action="store_true")
    a = ap.parse_args(argv)
    if a.command == "install":
        if not a.prefix:
            ap.error("install needs --prefix")
        print(install(a.prefix))
        return
    print(build(force=a.force, jobs=a.j, verbose=a.v))


if __name__ == "__main__":
    main()
