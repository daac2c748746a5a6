"""Builds libmdx.so (the HIP kernels + C ABI) for gfx950 with hipcc, and mdx/_host.so (the host
side of the Python functions, a CPython extension module on top of it) with g++, in-tree.

Usage: python build.py
Both land in the Python package (mdx/) so that they travel with the source tree;
nothing is installed.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
OBJ = ROOT / "build"
LIB = ROOT / "mdx" / "libmdx.so"
HOST = ROOT / "mdx" / "_host.so"

SOURCES = ["mdx_api.hip", "store_kvcache.hip", "unmask.hip", "logit_filter.hip", "filtered_pick.hip", "staircase_attn.hip", "staircase_attn_f32.hip", "paged_attn.hip", "paged_attn_f32.hip", "paged_attn_static.hip", "qk_norm_rope_store.hip", "layer_ops.hip", "linear.hip", "block_state.hip", "lm_head_unmask.hip", "lm_head_rows.hip", "calib_probe.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # hipcc -O3 forms packed fp32 ops on its own; they are kept out of every kernel here.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes",
]


def _compile(src: str) -> Path:
    obj = OBJ / (src.rsplit(".", 1)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", str(CSRC / src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l and l.strip() != "1 warning generated when compiling for host.")
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def _compile_host() -> Path:
    """host_ops.cpp -> build/host_ops.o: C++ against the headers of the installed torch, no device code."""
    import sysconfig
    from torch.utils.cpp_extension import include_paths
    obj = OBJ / "host_ops.o"
    includes = [f"-I{p}" for p in [*include_paths("cuda"), sysconfig.get_paths()["include"]]]
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           *(i.replace("-I", "-isystem", 1) for i in includes), "-c", str(CSRC / "host_ops.cpp"), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on host_ops.cpp:\n{r.stderr}")
    if r.stderr.strip():
        print(r.stderr, file=sys.stderr)
    return obj


def _link_host(obj: Path) -> None:
    """mdx/_host.so on libmdx.so (found next to it) and torch's libraries (loaded by then: torch is imported first)."""
    from torch.utils.cpp_extension import library_paths
    libs = library_paths("cuda")[0]
    cmd = ["g++", "-shared", "-o", str(HOST), str(obj), f"-L{LIB.parent}", "-l:libmdx.so", f"-L{libs}", "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{libs}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of _host.so failed:\n{r.stderr}")


def build_all(verbose: bool = True) -> Path:
    """Compiles every HIP source and links libmdx.so; always recompiles."""
    OBJ.mkdir(exist_ok=True)
    srcs = [s for s in SOURCES if (CSRC / s).exists()]
    missing = [s for s in SOURCES if not (CSRC / s).exists()]
    if missing:
        raise RuntimeError(f"missing sources: {missing}")
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, srcs))
        host_obj = host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    _link_host(host_obj)
    if verbose:
        print(f"built {LIB} ({LIB.stat().st_size} bytes) from {len(srcs)} sources, and {HOST.name}")
    return LIB


if __name__ == "__main__":
    build_all()
