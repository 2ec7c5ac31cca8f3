"""Build libomni_dit_hip.so for gfx950 with hipcc (cross-compiles without a GPU).

Usage:  python vllm-omni_amd/csrc/build.py [--force] [--jobs N]

Every translation unit is compiled to an object under csrc/build/ and linked into
``<package>/libomni_dit_hip.so`` next to the Python sources, so the library travels with the tree. The native host
path (``native.cpp``: host code against torch's headers, no device code) becomes ``<package>/_native.so``, a Python
extension module linked against that library.
"""

from __future__ import annotations

import argparse
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

CSRC = Path(__file__).resolve().parent
PKG = CSRC.parent
LIB_NAME = "libomni_dit_hip.so"
LIB_PATH = PKG / LIB_NAME
# bench.py's calibration probe (a bare MFMA loop): a library of its own, not part of the product's C ABI
PROBE_LIB_PATH = PKG / "libomni_dit_probe.so"
NATIVE_SRC = CSRC / "native.cpp"
NATIVE_PATH = PKG / "_native.so"
OBJ_DIR = CSRC / "build"
HEADERS = [CSRC / "odit_common.h", CSRC / "attn_common.h", CSRC / "attn_tail.h", CSRC / "gemm_bf16.h",
           CSRC / "gemm_epilogue.h", CSRC / "gemm_tile.h",
           CSRC / "gemm_heads.h", CSRC / "gemm_small.h", CSRC / "time_sinusoid.h", CSRC / "time_tokens.h", PKG.parent / "include" / "omni_dit.h"]

# (source file, extra defines, object stem)
UNITS: list[tuple[str, list[str], str]] = [
    ("api.hip", [], "api"),
    ("adaln.hip", [], "adaln"),
    ("pointwise.hip", [], "pointwise"),
    ("rel_l1.hip", [], "rel_l1"),
    ("qknorm_rope.hip", ["-DODIT_QK_TU=0"], "qknorm_rope_bf16"),
    ("qknorm_rope.hip", ["-DODIT_QK_TU=1"], "qknorm_rope_f16"),
    ("qknorm_rope.hip", ["-DODIT_QK_TU=2"], "qknorm_rope_f32"),
    ("attn_fwd.hip", [], "attn_fwd"),
    ("attn_fwd_dma.hip", [], "attn_fwd_dma"),
    ("linear.hip", [], "linear"),
    ("linear_few.hip", [], "linear_few"),
    ("linear_head.hip", [], "linear_head"),
    ("step.hip", [], "step"),
    ("time_tokens.hip", [], "time_tokens"),
    ("gemm_bf16.hip", [], "gemm_bf16"),
    ("gemm_bf16_tile.hip", [], "gemm_bf16_tile"),
    ("gemm_tile_heads.hip", [], "gemm_tile_heads"),
    ("gemm_tile_unless.hip", [], "gemm_tile_unless"),
    ("gemm_tile_apart.hip", [], "gemm_tile_apart"),
    ("gemm_tile_shared.hip", [], "gemm_tile_shared"),
    ("gemm_small.hip", [], "gemm_small"),
    ("gemm_small_heads.hip", [], "gemm_small_heads"),
    ("gemm_small_norm.hip", [], "gemm_small_norm"),
]
PROBE_UNITS: list[tuple[str, list[str], str]] = [("probe.hip", [], "probe")]

# the dense projections call hipBLASLt (its MFMA GEMM kernels); everything else is self-contained
LINK_LIBS = ["-L/opt/rocm/lib", "-lhipblaslt"]

# -packed-fp32-ops is switched off on purpose: v_pk_*_f32 forms are not trusted on this target.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found (looked on PATH and in /opt/rocm/bin)")
    return exe


def _stale(obj: Path, deps: list[Path]) -> bool:
    if not obj.exists():
        return True
    t = obj.stat().st_mtime
    return any(d.stat().st_mtime > t for d in deps)


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature; that line is noise
    err = "\n".join(l for l in proc.stderr.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{proc.stdout}\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")


def _native_compile(obj: Path) -> list[str]:
    """The host compiler's command for native.cpp (torch's and Python's headers; no offload)."""
    import sysconfig

    import torch

    inc = Path(torch.__file__).resolve().parent / "include"
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
            "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-isystem{inc}",
            f"-isystem{inc / 'torch' / 'csrc' / 'api' / 'include'}", "-isystem/opt/rocm/include",
            f"-isystem{sysconfig.get_paths()['include']}", "-c", str(NATIVE_SRC), "-o", str(obj)]


def _native_link(obj: Path, out: Path) -> list[str]:
    import torch

    lib = Path(torch.__file__).resolve().parent / "lib"
    return [os.environ.get("CXX", "g++"), "-shared", "-o", str(out), str(obj), f"-L{PKG}", "-l:" + LIB_NAME, f"-L{lib}",
            "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]


def build(force: bool = False, jobs: int | None = None, verbose: bool = True) -> Path:
    hipcc = _hipcc()
    OBJ_DIR.mkdir(exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    work = []
    objs: dict[Path, list[Path]] = {LIB_PATH: [], PROBE_LIB_PATH: []}
    for lib, units in ((LIB_PATH, UNITS), (PROBE_LIB_PATH, PROBE_UNITS)):
        for src, defines, stem in units:
            src_path = CSRC / src
            if not src_path.exists():
                raise RuntimeError(f"missing source {src_path}")
            obj = OBJ_DIR / f"{stem}.o"
            objs[lib].append(obj)
            if force or _stale(obj, [src_path, *HEADERS, Path(__file__)]):
                work.append([hipcc, *HIPCC_FLAGS, *defines, "-c", str(src_path), "-o", str(obj)])
    native_obj = OBJ_DIR / "native.o"
    native_stale = force or _stale(native_obj, [NATIVE_SRC, PKG.parent / "include" / "omni_dit.h", Path(__file__)])
    host = [_native_compile(native_obj)] if native_stale else []
    if verbose:
        print(f"[omni_dit build] compiling {len(work) + len(host)}/{len(UNITS) + len(PROBE_UNITS) + 1} units with {jobs} jobs", flush=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        list(ex.map(_run, host + work))
    for lib, link in ((LIB_PATH, LINK_LIBS), (PROBE_LIB_PATH, [])):
        if work or force or not lib.exists():
            tmp = lib.with_suffix(".so.tmp")
            _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs[lib]), *link])
            os.replace(tmp, lib)
        if verbose:
            print(f"[omni_dit build] {lib} ({lib.stat().st_size} bytes)", flush=True)
    if native_stale or not NATIVE_PATH.exists():
        tmp = NATIVE_PATH.with_suffix(".so.tmp")
        _run(_native_link(native_obj, tmp))
        os.replace(tmp, NATIVE_PATH)
    if verbose:
        print(f"[omni_dit build] {NATIVE_PATH} ({NATIVE_PATH.stat().st_size} bytes)", flush=True)
    return LIB_PATH


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--jobs", type=int, default=None)
    a = ap.parse_args()
    build(force=a.force, jobs=a.jobs)
