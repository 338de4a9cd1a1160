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
    return LIB_PATH


def ensure_built():
    """For test sessions, the smoke test and the benchmark: builds the library when it is not there (the package itself
    never does: it raises)."""
    lib = os.path.join(LIB_DIR, "libe3x.so")
    if not os.path.exists(lib):
        build_library(verbose=False, force=False)
    return lib


if __name__ == "__main__":
    build_library(verbose=True, force="--incremental" not in sys.argv)
    print("built", LIB_PATH)
