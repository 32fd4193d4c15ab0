"""Build libjigsaw_hip.so (gfx950) from the HIP sources under ``csrc/`` and, against it and
torch, the native host module ``_host.so`` from ``csrc/host.cpp``.

Usage: ``python -m jigsaw_amd.build [--jobs N] [--force]``. hipcc cross-compiles
for gfx950 without a GPU present. Objects go to ``csrc/build/``, the library to
``lib/libjigsaw_hip.so``, the module to ``_host.so`` (all git-ignored; the built files travel with the tree).
"""

from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
OBJ = CSRC / "build"
LIB = ROOT / "lib" / "libjigsaw_hip.so"
HOST = ROOT / "_host.so"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    # Packed-fp32 VALU forms are kept out of the generated code on purpose.
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
]


# Kernels whose vector instructions read or scale their matrix accumulators (softmax on the scores, the
# running rescale, epilogues) keep the accumulators in ordinary vector registers: left to its default the
# compiler puts them in the accumulation registers and moves them over and back with v_accvgpr_read /
# v_accvgpr_write around every such use (64 moves per loop iteration in the wide attention forward).
PER_FILE_FLAGS = {
    name: ["-mllvm", "-amdgpu-mfma-vgpr-form"]
    for name in ("attn_wide.hip", "attn_swin.hip", "attn_window.hip", "attn_f32_mfma.hip", "conv_f32.hip", "proj_mfma.hip")
}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found; set HIPCC or install ROCm under /opt/rocm")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _newer(a: Path, deps: list[Path]) -> bool:
    if not a.exists():
        return False
    t = a.stat().st_mtime
    return all(d.stat().st_mtime <= t for d in deps)


def _compile(src: Path, force: bool, extra: list[str]) -> Path:
    obj = OBJ / (src.stem + ".o")
    deps = [src, *CSRC.glob("*.h"), ROOT.parent / "include" / "jigsaw_hip.h"]
    if not force and _newer(obj, deps):
        return obj
    cmd = [hipcc(), *HIPCC_FLAGS, *PER_FILE_FLAGS.get(src.name, []), *extra, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the packed-fp32 feature and says so; harmless.
    err = "\n".join(
        ln for ln in proc.stderr.splitlines() if "packed-fp32-ops" not in ln
    )
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _run(cmd: list[str], what: str) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{proc.stderr}")


def _compile_host(force: bool) -> Path:
    """Object of ``csrc/host.cpp`` (no device code: the host compiler takes it)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    src, obj = CSRC / "host.cpp", OBJ / "host.o"
    if not force and _newer(obj, [src, ROOT.parent / "include" / "jigsaw_hip.h"]):
        return obj
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-DTORCH_EXTENSION_NAME=_host",
           "-DTORCH_API_INCLUDE_EXTENSION_H", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM"]  # (for the stream's type in c10/hip)
    for path in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"], str(Path(hipcc()).resolve().parent.parent / "include")):
        cmd += ["-isystem", path]
    _run([*cmd, "-c", str(src), "-o", str(obj)], "g++ host.cpp")
    return obj


def _link_host(obj: Path) -> None:
    from torch.utils import cpp_extension

    cmd = ["g++", "-shared", "-o", str(HOST), str(obj), f"-L{LIB.parent}", "-ljigsaw_hip", "-Wl,-rpath,$ORIGIN/lib"]
    for path in cpp_extension.library_paths():
        cmd += [f"-L{path}", f"-Wl,-rpath,{path}"]
    _run([*cmd, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"], "link of _host.so")


def build(jobs: int = 8, force: bool = False, extra: list[str] | None = None) -> Path:
    """Compile every ``csrc/*.hip`` and link ``lib/libjigsaw_hip.so``; compile and link ``_host.so``."""
    extra = list(extra or [])
    OBJ.mkdir(parents=True, exist_ok=True)
    LIB.parent.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as pool:
        host = pool.submit(_compile_host, force)
        objs = list(pool.map(lambda s: _compile(s, force, extra), srcs))
        host_obj = host.result()
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(LIB)]
    cmd += [str(o) for o in objs]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    _link_host(host_obj)
    return LIB


def main() -> None:
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--jobs", type=int, default=min(8, os.cpu_count() or 1))
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--save-temps", action="store_true", help="keep ISA under csrc/build/")
    ns = ap.parse_args()
    extra = ["-save-temps=obj"] if ns.save_temps else []
    print(build(ns.jobs, ns.force, extra))


if __name__ == "__main__":
    main()
