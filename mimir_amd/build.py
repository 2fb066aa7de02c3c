"""Build libmimir_prefixlm.so (the C-ABI HIP library) and the native host calls in-tree for gfx950.

Every HIP source under ``mimir_amd/csrc`` is compiled with hipcc for
``--offload-arch=gfx950`` and linked into ``mimir_amd/_lib/libmimir_prefixlm.so``.
No torch extension machinery is involved: the library exports only the
``extern "C"`` entry points declared in ``include/mimir_prefixlm.h`` and is loaded
with ctypes.  ``csrc/host_calls.cpp`` (no device code; g++ and torch's C++ headers) becomes
``mimir_amd/_lib/_host_calls.so``, the Python module that makes the common calls; the package
works without it.  Run ``python -m mimir_amd.build`` (or ``__graft_entry__.build()``).
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_DIR = PKG_DIR / "_lib"
LIB_PATH = LIB_DIR / "libmimir_prefixlm.so"
HOST_SOURCE = CSRC / "host_calls.cpp"
HOST_PATH = LIB_DIR / "_host_calls.so"
ARCH = "gfx950"

# Packed FP32 (v_pk_*_f32) is disabled: hipcc otherwise forms them from float2
# arithmetic.  The host pass warns that it does not know the feature; harmless.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]

# Per-source code generation options (none at present).
SOURCE_FLAGS: dict = {}

SOURCES = [
    "prefixlm_capi.hip",
    "prefixlm_fwd_bf16.hip",
    "prefixlm_bwd_bf16.hip",
    "prefixlm_bwd_dq_bf16.hip",
    "prefixlm_bwd_dq_ds_bf16.hip",
    "prefixlm_bwd_dkdv_bf16.hip",
    "prefixlm_bwd_dkdv_pair_bf16.hip",
    "prefixlm_f32.hip",
    "prefixlm_prologue.hip",
    "prefixlm_layer.hip",
    "prefixlm_cache_bf16.hip",
    "prefixlm_noalloc.hip",
]


def hipcc() -> str:
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cand = Path(rocm) / "bin" / "hipcc"
    if cand.exists():
        return str(cand)
    found = shutil.which("hipcc")
    if not found:
        raise RuntimeError("hipcc not found; set ROCM_PATH")
    return found


def _compile(src: Path, obj: Path) -> None:
    cmd = [hipcc(), *HIPCC_FLAGS, *SOURCE_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)


def _build_host() -> None:
    """Compile the native host calls against the running Python and torch.

    They only shorten calls that the general path in Python makes as well, so a
    machine without a C++ compiler or Python's headers still gets the library."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    libs = Path(torch.__file__).resolve().parent / "lib"
    tmp = HOST_PATH.with_suffix(".so.tmp")
    args = ["-O2", "-std=c++17", "-fPIC", "-shared",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            f'-DMIMIR_BUILT_FOR="torch {torch.__version__}, Python {sys.version_info[0]}.{sys.version_info[1]}"',
            *(x for p in include_paths() for x in ("-isystem", p)), f"-I{sysconfig.get_paths()['include']}",
            str(HOST_SOURCE), "-o", str(tmp), f"-L{libs}", f"-Wl,-rpath,{libs}", "-ltorch_python", "-ltorch_cpu", "-lc10"]
    try:
        res = subprocess.run([os.environ.get("CXX", "g++"), *args], capture_output=True, text=True)
        error = res.stderr if res.returncode != 0 else ""
    except OSError as e:
        error = str(e)
    if error:
        HOST_PATH.unlink(missing_ok=True)  # not one of other sources
        print(f"warning: {HOST_SOURCE.name} was not compiled, calls will take the general path:\n{error}", file=sys.stderr)
    else:
        os.replace(tmp, HOST_PATH)


def build(verbose: bool = True) -> Path:
    """Compile every source and link the shared library; returns its path."""
    obj_dir = LIB_DIR / "obj"
    obj_dir.mkdir(parents=True, exist_ok=True)
    objs = [obj_dir / (s.rsplit(".", 1)[0] + ".o") for s in SOURCES]
    with ThreadPoolExecutor(max_workers=min(4, len(SOURCES))) as ex:
        host = ex.submit(_build_host)
        list(ex.map(lambda so: _compile(CSRC / so[0], so[1]), zip(SOURCES, objs)))
        host.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    build()
