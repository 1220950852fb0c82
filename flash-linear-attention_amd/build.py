"""Build libfla_hip.so (gfx950) from csrc/*.hip with hipcc, and the host extension _fla_host.so from csrc/torch_host.cpp
with g++, in-tree.

    python flash-linear-attention_amd/build.py [--force] [-j N]

Each translation unit is compiled to an object file under ``build/`` (kept out
of version control) and the objects are linked into ``fla_amd/lib/libfla_hip.so``.
hipcc cross-compiles, so this runs without a GPU.
"""
import argparse
import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "build")
LIB_DIR = os.path.join(HERE, "fla_amd", "lib")
LIB_PATH = os.path.join(LIB_DIR, "libfla_hip.so")
HOST_SRC, HOST_PATH = os.path.join(CSRC, "torch_host.cpp"), os.path.join(LIB_DIR, "_fla_host.so")

HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17",
    # packed fp32 VALU forms are kept off
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
# Keeps MFMA accumulators in ordinary vector registers: elementwise work on them (decay, scaling,
# conversion for stores) then needs no copies out of and back into the accumulation registers.
# Only where it measured faster (gdr_bwd_dhu 216 -> 204 us, gla_bwd_dh 166 -> 162 us); the forward state
# scans lose with it.
VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
VGPR_FORM_SOURCES = {"gdr_bwd.hip", "gdr_bwd_chunk.hip", "gdr_bwd_scan.hip", "gla_bwd.hip", "gla_bwd_chunk.hip"}


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _newest_header():
    hdrs = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    hdrs.append(os.path.join(HERE, "..", "include", "fla_hip.h"))
    return max(os.path.getmtime(h) for h in hdrs)


def _compile(src, force):
    obj = os.path.join(OBJ_DIR, src[:-4] + ".o")
    path = os.path.join(CSRC, src)
    if (not force and os.path.exists(obj)
            and os.path.getmtime(obj) >= max(os.path.getmtime(path), _newest_header())):
        return obj, ""
    cmd = [HIPCC] + FLAGS + (VGPR_FORM if src in VGPR_FORM_SOURCES else []) + ["-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    log = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                    if "not a recognized feature" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{log}")
    return obj, log


def _build_host(force):
    """The CPython extension over libfla_hip.so (host code only; torch is asked for its include and library folders)."""
    import torch
    from torch.utils import cpp_extension as ext
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    includes = [p for p in ext.include_paths() if os.path.isdir(p)] + [os.path.join(rocm, "include"), "/opt/rocm/include",
                                                                       sysconfig.get_path("include")]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"]
    for p in includes:
        cmd += ["-isystem", p]
    cmd += [HOST_SRC, "-o", HOST_PATH]
    for p in ext.library_paths():
        cmd += ["-L" + p]
    cmd += ["-L" + LIB_DIR, "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-lfla_hip",
            "-Wl,-rpath,$ORIGIN"]
    # Up to date: newer than its sources and built by this very command against this torch, whose C++ interface changes
    # from version to version without a file here becoming newer.
    stamp = os.path.join(OBJ_DIR, "_fla_host.stamp")
    built_for = "\n".join([torch.__version__, str(torch.version.git_version)] + cmd)
    header = os.path.join(HERE, "..", "include", "fla_hip.h")
    if (not force and os.path.exists(HOST_PATH) and os.path.exists(stamp)
            and os.path.getmtime(HOST_PATH) >= max(os.path.getmtime(HOST_SRC), os.path.getmtime(header))):
        with open(stamp) as f:
            if f.read() == built_for:
                return ""
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed on torch_host.cpp:\n" + r.stdout + r.stderr)
    with open(stamp, "w") as f:
        f.write(built_for)
    return r.stderr


def build(force=False, jobs=None, verbose=True):
    os.makedirs(OBJ_DIR, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        results = list(ex.map(lambda s: _compile(s, force), sources()))
    objs = [o for o, _ in results]
    for _, log in results:
        if log.strip() and verbose:
            print(log)
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    _build_host(force)
    if verbose:
        print(f"built {LIB_PATH} from {len(objs)} objects, and {HOST_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("-j", type=int, default=None)
    a = ap.parse_args()
    try:
        build(force=a.force, jobs=a.j)
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
