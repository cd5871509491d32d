"""Build recipe of the two native pieces: libslapo_amd.so (hipcc cross-compiles every csrc/*.hip
for gfx950) and the extension module _host.so (g++ compiles csrc/host_ops.cpp against torch's
headers; it calls the kernels through the C ABI of the library beside it).

Both are built in-tree (slapo_amd/) so that they travel with the source tree; nothing is compiled
at import time.  `python -m slapo_amd.build` rebuilds them.
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC_DIR = os.path.join(PKG_DIR, "csrc")
OBJ_DIR = os.path.join(CSRC_DIR, "build")
LIB_PATH = os.path.join(PKG_DIR, "libslapo_amd.so")
HOST_PATH = os.path.join(PKG_DIR, "_host.so")

ARCH = "gfx950"

# -packed-fp32-ops is switched off on purpose: the compiler must not form v_pk_*_f32.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=fast",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Wno-unknown-attributes",
]


# The MFMA attention kernels never compute with NaNs on their defined paths (masked scores are
# -inf, guarded before every subtraction); telling the compiler so removes the canonicalising
# v_max x,x it would otherwise put in front of every max of an MFMA result.
PER_FILE_FLAGS = {
    "attn_fwd_f16.hip": ["-fno-honor-nans"],
    "attn_fwd_bf16.hip": ["-fno-honor-nans"],
    "attn_bwd_f16.hip": ["-fno-honor-nans"],
    "attn_bwd_bf16.hip": ["-fno-honor-nans"],
    "attn_bwd_dq_f16.hip": ["-fno-honor-nans"],
    "attn_bwd_dq_bf16.hip": ["-fno-honor-nans"],
    "attn_bwd_both_f16.hip": ["-fno-honor-nans"],
    "attn_bwd_both_bf16.hip": ["-fno-honor-nans"],
}


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libslapo_amd.so cannot be built")
    return exe


def sources() -> list[str]:
    return sorted(
        os.path.join(CSRC_DIR, f) for f in os.listdir(CSRC_DIR) if f.endswith(".hip")
    )


def _compile_one(src: str, extra: list[str]) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + ".o")
    per_file = PER_FILE_FLAGS.get(os.path.basename(src), [])
    cmd = [_hipcc(), *HIPCC_FLAGS, *per_file, *extra, "-c", src, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{proc.stdout}\n{proc.stderr}")
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_host() -> str:
    """Object file of the extension module: host code only, no device pass."""
    from torch.utils.cpp_extension import include_paths

    obj = os.path.join(OBJ_DIR, "host_ops.o")
    dirs = [*include_paths(), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM", *[f for d in dirs for f in ("-isystem", d)], "-c",
           os.path.join(CSRC_DIR, "host_ops.cpp"), "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed for host_ops.cpp:\n{proc.stdout}\n{proc.stderr}")
    return obj


def _link_host(obj: str) -> str:
    """torch's libraries are loaded by `import torch` before the module is; libslapo_amd.so is found
    beside it."""
    from torch.utils.cpp_extension import library_paths

    tmp = HOST_PATH + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, f"-L{PKG_DIR}", "-lslapo_amd",
           *[f"-L{d}" for d in library_paths()], "-ltorch_python", "-ltorch", "-ltorch_cpu",
           "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, HOST_PATH)
    return HOST_PATH


def build_library(verbose: bool = False, extra_flags: list[str] | None = None) -> str:
    """Compile all kernels and the host module and link both; always recompiles."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    extra = list(extra_flags or [])
    srcs = sources()
    if verbose:
        print(f"[slapo_amd.build] compiling {len(srcs)} files for {ARCH}", flush=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as pool:
        host_obj = pool.submit(_compile_host)
        objs = list(pool.map(lambda s: _compile_one(s, extra), srcs))
    tmp = LIB_PATH + ".tmp"
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host(host_obj.result())
    if verbose:
        print(f"[slapo_amd.build] wrote {LIB_PATH} and {HOST_PATH}", flush=True)
    return LIB_PATH


if __name__ == "__main__":
    build_library(verbose=True)
