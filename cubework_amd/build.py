"""Build libcubework_hip.so (the gfx950 kernels + C ABI), libcubework_diag.so (measurement aids that only
bench.py and their tests load) with hipcc and _host.so (the operators' native host side) with g++, in-tree.

    python -m cubework_amd.build          # compile every source, link all three

hipcc cross-compiles for gfx950 without a GPU. The libraries are written next to
this file so that they travel with the source tree.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(CSRC, "build")
LIB_PATH = os.path.join(HERE, "libcubework_hip.so")

# compiled once per (element type, orientation, tile height) and (element type, orientation, configuration)
TILE_OBJECTS = ["%s.hip:%s:%s:%d" % (src, e, layout, cfg) for src, cfgs in (("gemm_wide", (256, 224, 192, 160, 128, 2192, 2160, 2128)), ("gemm_tile", (1, 2, 3, 4)))
                for cfg in cfgs for layout in ("NN", "NT", "TN") for e in ("bf16_t", "f16_t") if cfg < 2000 or layout != "TN"]
SOURCES = TILE_OBJECTS + [  # slowest first
    "gemm_bf16_tn.hip", "gemm_f16_tn.hip", "gemm_bf16_nn.hip", "gemm_f16_nn.hip", "gemm_bf16_nt.hip", "gemm_f16_nt.hip",
    "cw_runtime.hip", "cw_api.hip", "gemm_plan.hip", "gemm_bf16.hip", "gemm_f32.hip", "epilogue.hip", "layernorm.hip", "vpce.hip",
    "attention.hip", "attention_bwd.hip", "embedding.hip", "embed_sort.hip", "clip_grad.hip", "cast.hip"]
# the measurement library: its own kernels plus the runtime services (error text, device check), nothing else
DIAG_SOURCES = ["diag_gemm.hip", "diag.hip"]
DIAG_LIB_PATH = os.path.join(HERE, "libcubework_diag.so")

# the operators' native host side: a Python extension on torch's C++ API
HOST_SOURCES = ["host_ops.cpp", "host_nodes.cpp"]
HOST_PATH = os.path.join(HERE, "_host.so")

# Packed-fp32 VALU forms are kept off: plain float code only.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Wno-unknown-warning-option",
]


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _compile(src, extra=(), obj_dir=None):
    src, *variant = src.split(":")
    obj = os.path.join(obj_dir or OBJ_DIR, "_".join([os.path.splitext(src)[0], *variant]) + ".o")
    defines = ["-D%s=%s" % kv for kv in zip(("CW_TILE_E", "CW_TILE_LAYOUT", "CW_TILE_CFG"), variant)]
    cmd = [_hipcc(), *HIPCC_FLAGS, *extra, *defines, "-c", os.path.join(CSRC, src), "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s\n%s" % (src, proc.stdout, proc.stderr))
    return obj


def build_host(verbose=True):
    """Compile and link the host extension (host compiler only; it holds no device code)."""
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    include = [os.path.join(os.path.dirname(HERE), "include"), os.path.join(root, "include"),
               os.path.join(root, "include", "torch", "csrc", "api", "include"), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    tmp = HOST_PATH + ".tmp"
    cxx = [os.environ.get("CXX", "g++")]
    flags = ["-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
             "-DTORCH_EXTENSION_NAME=_host", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, *["-I" + d for d in include]]
    objs = [os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".host.o") for src in HOST_SOURCES]

    def run(cmd):
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError("host extension failed:\n%s\n%s" % (proc.stdout, proc.stderr))

    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(len(HOST_SOURCES)) as pool:
        list(pool.map(lambda pair: run([*cxx, *flags, "-c", os.path.join(CSRC, pair[0]), "-o", pair[1]]), zip(HOST_SOURCES, objs)))
    run([*cxx, "-shared", *objs, "-o", tmp, "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python"])
    os.replace(tmp, HOST_PATH)
    if verbose:
        print("built", HOST_PATH, os.path.getsize(HOST_PATH), "bytes")


def build(verbose=True, extra_flags=(), lib_path=None, obj_dir=None):
    """Compile every HIP source for gfx950 and link the shared library.
    extra_flags / lib_path / obj_dir build a variant beside the default one."""
    lib_path = lib_path or LIB_PATH
    obj_dir = obj_dir or OBJ_DIR
    os.makedirs(obj_dir, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
        host = pool.submit(build_host, verbose) if lib_path == LIB_PATH else None
        objs = list(pool.map(lambda src: _compile(src, extra_flags, obj_dir), SOURCES + DIAG_SOURCES))
    if host is not None:
        host.result()
    by_src = dict(zip(SOURCES + DIAG_SOURCES, objs))

    def link(members, path):
        tmp = path + ".tmp"
        cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *[by_src[m] for m in members], "-o", tmp]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError("link failed:\n%s\n%s" % (proc.stdout, proc.stderr))
        os.replace(tmp, path)
        if verbose:
            print("built", path, os.path.getsize(path), "bytes")

    link(SOURCES, lib_path)
    diag_path = DIAG_LIB_PATH if lib_path == LIB_PATH else os.path.splitext(lib_path)[0] + "_diag.so"
    link(DIAG_SOURCES + ["cw_runtime.hip"], diag_path)
    return lib_path


if __name__ == "__main__":
    build()
    sys.exit(0)
