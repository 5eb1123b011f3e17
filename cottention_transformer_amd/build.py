"""Builds libcottention_hip.so for gfx950 with hipcc (cross-compiles without a GPU), and the native host module.

Every output is written under a name of its own and moved into place whole, so processes that build at the same time never
see each other's halves.

    python -m cottention_transformer_amd.build            # compile every translation unit and link
"""
import glob
import hashlib
import os
import subprocess
import sys
import uuid
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "build", "obj")
LIB_PATH = os.path.join(HERE, "lib", "libcottention_hip.so")

SOURCES = ["cott_api.hip", "cott_mfma_bf16.hip", "cott_mfma_fp16.hip", "cott_mfma_f32.hip", "cott_generic.hip", "cott_wide.hip", "cott_decode_block.hip", "cott_prep.hip", "cott_block.hip", "cott_calib.hip"]

# -packed-fp32-ops off: scalar/float2 fp32 code must not be fused into v_pk_*_f32 instructions.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return "hipcc"


def _run_to(path, cmd, what):
    """Run a compiler or linker that writes its last argument, `path`; returns what it printed."""
    tmp = f"{path}.{uuid.uuid4().hex}.tmp"
    try:
        res = subprocess.run(cmd + [tmp], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"{what}:\n{res.stdout}")
        os.replace(tmp, path)
    finally:
        if os.path.exists(tmp):
            os.unlink(tmp)
    return res.stdout


def _compile(src):
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    printed = _run_to(obj, [hipcc()] + HIPCC_FLAGS + ["-c", os.path.join(CSRC, src), "-o"], f"hipcc failed on {src}")
    return obj, "\n".join(l for l in printed.splitlines() if "packed-fp32-ops" not in l)


def native_path():
    """Where the native host module for this torch, this Python and this csrc/native.cpp lies.  It reads torch's objects through
    inlined accessors, so a file built against another torch could misread them; its name says what it was built from."""
    import torch
    with open(os.path.join(CSRC, "native.cpp"), "rb") as f:
        source = f.read()
    built_for = (torch.__version__, str(torch.version.git_version), str(torch._C._GLIBCXX_USE_CXX11_ABI), sys.version)
    tag = hashlib.sha256(b"\0".join([source, *(x.encode() for x in built_for)])).hexdigest()[:16]
    return os.path.join(HERE, f"_native.{tag}.so")


def build_native():
    """Compile the native host module (_native, csrc/native.cpp) against the installed torch; returns its path."""
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    path = native_path()
    _run_to(path, ["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden",
                   f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                   "-I" + os.path.join(root, "include"), "-I" + os.path.join(root, "include", "torch", "csrc", "api", "include"),
                   "-I" + sysconfig.get_paths()["include"], os.path.join(CSRC, "native.cpp"),
                   "-L" + os.path.join(root, "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-o"], "g++ failed on native.cpp")
    return path


def build_library(verbose=False, jobs=None):
    """Compile all HIP sources and link the shared library; returns its path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    os.makedirs(os.path.dirname(LIB_PATH), exist_ok=True)
    jobs = jobs or min(len(SOURCES), max(1, (os.cpu_count() or 2) // 2))
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        results = list(pool.map(_compile, SOURCES))
    if verbose:
        for _, out in results:
            if out.strip():
                print(out)
    objs = [o for o, _ in results]
    _run_to(LIB_PATH, [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o"], "link failed")
    return LIB_PATH


def build(verbose=False, jobs=None):
    """The shared library, then the native host module in place of older ones; returns the library's path."""
    path = build_library(verbose, jobs)
    native = build_native()
    for old in glob.glob(os.path.join(HERE, "_native*.so")):
        if old != native:
            os.unlink(old)
    return path


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
