"""Builds libe3x.so (gfx950) in-tree: python -m e3nn_amd.csrc.build

Every translation unit is compiled with hipcc; device code is built with packed-fp32
instruction selection disabled.  The device templates under templates/ are embedded
into the library as string constants so that the kernel specialiser needs no files at
run time.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB_DIR = os.path.join(PKG, "lib")
OBJ_DIR = os.path.join(HERE, "build")
LIB_PATH = os.path.join(LIB_DIR, "libe3x.so")
HOST_PATH = os.path.join(LIB_DIR, "_e3x_host.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

SOURCES = ["api.cpp", "wigner.cpp", "jit.cpp", "tp.cpp", "fc.cpp", "sh.hip", "graph.hip", "gate.hip"]
TEMPLATES = [("kTplCommon", "common.inc"), ("kTplPieces", "pieces.inc"), ("kTplUvu", "uvu.inc"), ("kTplUvuFc", "uvu_fc.inc"), ("kTplUvuRowgrad", "uvu_rowgrad.inc"), ("kTplUvuMfma", "uvu_mfma.inc"), ("kTplUvwSmall", "uvw_small.inc"),
             ("kTplUvwMfma", "uvw_mfma.inc"), ("kTplUvwMfmaBf16", "uvw_mfma_bf16.inc"), ("kTplUvwFew", "uvw_few.inc"), ("kTplUvwUnits", "uvw_units.inc"), ("kTplUvwMfmaHalf", "uvw_mfma_half.inc"),
             ("kTplUvwMfmaDw", "uvw_mfma_dw.inc"), ("kTplUvwDwWide", "uvw_dw_wide.inc"),
             ("kTplUvwNode", "uvw_node.inc"), ("kTplUvwNodeDw", "uvw_node_dw.inc"),
             ("kTplFcMfma", "fc_mfma.inc"), ("kTplFcDw", "fc_dw.inc")]
DEVICE_FLAGS = ["--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON_FLAGS = ["-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-Wno-unused-function", "-Wno-unused-result"]


def hipcc():
    return os.environ.get("E3X_HIPCC") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else "hipcc")


def _embed_templates():
    out = ['// generated by build.py from templates/*.inc', '#include "../jit.h"', "namespace e3x {"]
    for sym, name in TEMPLATES:
        path = os.path.join(HERE, "templates", name)
        text = open(path).read() if os.path.exists(path) else ""
        assert ')E3XTPL"' not in text
        out.append(f'const char* const {sym} = R"E3XTPL(\n{text})E3XTPL";')
    out.append("}  // namespace e3x")
    path = os.path.join(OBJ_DIR, "templates_embedded.cpp")
    text = "\n".join(out) + "\n"
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as f:
            f.write(text)
    return path


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # the host pass does not know the packed-fp32 target feature and says so: harmless
    lines = [l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l and "is not a recognized feature" not in l]
    if r.returncode != 0:
        raise RuntimeError("build failed:\n" + " ".join(cmd) + "\n" + r.stdout)
    if verbose and lines:
        print("\n".join(lines), flush=True)


def build_library(verbose=True, force=True):
    os.makedirs(LIB_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = [os.path.join(HERE, s) for s in SOURCES] + [_embed_templates()]
    deps = [os.path.join(HERE, f) for f in ("e3x_internal.h", "jit.h")] + [os.path.join(PKG, "..", "include", "e3x.h")]
    newest_dep = max(os.path.getmtime(d) for d in deps)
    objs = []
    for src in srcs:
        obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
        objs.append(obj)
        if not force and os.path.exists(obj) and os.path.getmtime(obj) > max(os.path.getmtime(src), newest_dep):
            continue
        cmd = [hipcc(), "-c", src, "-o", obj] + COMMON_FLAGS
        if src.endswith(".hip"):
            cmd += DEVICE_FLAGS
        else:
            cmd += ["-x", "hip", "--offload-host-only"] if False else []
        _run(cmd, verbose)
    # exports: the C ABI of include/e3x.h and nothing else (template instantiations of the standard library carry
    # default visibility whatever the compile flags say)
    vs = os.path.join(OBJ_DIR, "exports.map")
    with open(vs, "w") as f:
        f.write("{ global: e3x_*; local: *; };\n")
    _run([hipcc(), "-shared", "-o", LIB_PATH] + objs + ["-ldl", "-Wl,--version-script=" + vs], verbose)
    build_host(verbose, force)
    return LIB_PATH


def build_host(verbose=True, force=True):
    """The extension module of the host path, against libe3x.so and this interpreter's torch."""
    import sysconfig

    import torch

    src = os.path.join(HERE, "host.cpp")
    header = os.path.join(PKG, "..", "include", "e3x.h")
    if not force and os.path.exists(HOST_PATH) and os.path.getmtime(HOST_PATH) > max(os.path.getmtime(src), os.path.getmtime(header)):
        return
    torch_dir = os.path.dirname(torch.__file__)
    include = [os.path.join(torch_dir, "include"), os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"), ROCM + "/include",
               sysconfig.get_paths()["include"]]  # fmt: skip
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-DTORCH_EXTENSION_NAME=_e3x_host", "-DUSE_ROCM",
           "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]  # fmt: skip
    cmd += [a for d in include for a in ("-isystem", d)] + [src, "-o", HOST_PATH, "-L" + LIB_DIR, "-l:libe3x.so", "-L" + os.path.join(torch_dir, "lib")]
    _run(cmd + ["-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-ltorch_python", "-Wl,-rpath,$ORIGIN"], verbose)


def ensure_built():
    """For test sessions, the smoke test and the benchmark: builds the library when it is not there (the package itself
    never does: it raises)."""
    lib = os.path.join(LIB_DIR, "libe3x.so")
    if not (os.path.exists(lib) and os.path.exists(HOST_PATH)):
        build_library(verbose=False, force=False)
    return lib


if __name__ == "__main__":
    build_library(verbose=True, force="--incremental" not in sys.argv)
    print("built", LIB_PATH)
