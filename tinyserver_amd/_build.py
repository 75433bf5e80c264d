"""Build libtsa.so, the gfx950 HIP library behind the C ABI in include/tsa_api.h,
and _tsa_host.so, the Python extension that calls it with torch tensors.

Every HIP source is compiled with hipcc for gfx950 only, in parallel, into
tinyserver_amd/_build/, and linked in place as tinyserver_amd/libtsa.so so the
library travels with the source tree; the extension is one host C++ file,
built beside it. Run ``python -m tinyserver_amd._build``.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libtsa.so"
HOST = PKG / "_tsa_host.so"
SOURCES = ["tsa_common.hip", "kv_store.hip", "qk_norm_rope.hip", "paged_decode.hip", "paged_decode_f32.hip",
           "varlen_prefill.hip", "varlen_prefill_w64.hip", "varlen_prefill_f32.hip", "sampling.hip"]
ARCH = "gfx950"
# Packed-fp32 VALU instructions are disabled: the compiler may not form them.
CFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; the HIP library cannot be built")
    return path


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "packed-fp32-ops"  # the host pass does not know the feature; harmless
    err = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{err}")
    if err.strip():
        print(err, file=sys.stderr)


def _host_cmd(obj: Path) -> list[str]:
    import torch
    from torch.utils.cpp_extension import include_paths

    return ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{ROOT / 'include'}",
            *(f"-isystem{p}" for p in include_paths()), f"-isystem{sysconfig.get_path('include')}", "-c",
            str(CSRC / "host_call.cpp"), "-o", str(obj)]


def build(verbose: bool = False) -> Path:
    """Compile every HIP source for gfx950 and link libtsa.so, then the host
    extension. Always rebuilds."""
    BUILD.mkdir(exist_ok=True)
    cc = hipcc()
    objs = [BUILD / (Path(s).stem + ".o") for s in SOURCES]

    def compile_one(src_obj):
        src, obj = src_obj
        if src == "host_call.cpp":
            return _run(_host_cmd(obj))
        cmd = [cc, *CFLAGS, "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)

    host_obj = BUILD / "host_call.o"
    jobs = min(len(SOURCES) + 1, int(os.environ.get("MAX_JOBS", os.cpu_count() or 4)))
    with ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        list(ex.map(compile_one, [*zip(SOURCES, objs), ("host_call.cpp", host_obj)]))
    tmp = LIB.with_suffix(".so.tmp")
    _run([cc, f"--offload-arch={ARCH}", "-shared", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, LIB)
    import torch

    libs = Path(torch.__file__).resolve().parent / "lib"
    tmp = HOST.with_suffix(".so.tmp")
    _run(["g++", "-shared", "-o", str(tmp), str(host_obj), f"-L{PKG}", "-ltsa", f"-L{libs}", "-ltorch_python",
          "-ltorch_cpu", "-lc10", "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{libs}"])
    os.replace(tmp, HOST)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
