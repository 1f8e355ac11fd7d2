"""Builds libtrida_hip.so (every csrc/*.hip, gfx950) in-tree with hipcc.

    python -m trida_stack_amd.build          # compile + link
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OBJ = PKG / "_build"
LIB = PKG / "libtrida_hip.so"
ARCH = os.environ.get("TRIDA_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
    # packed fp32 VALU ops stay off: the compiler emits plain v_fma/v_mul instead
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{PKG.parent / 'include'}",
]

# attention.hip: MFMA accumulators in the ordinary registers. Its kernels of head dim 256 hold more than 256 registers,
# for which the compiler would keep the accumulators in the accumulation half and move them at every rescale and
# loop edge (about 400 moves a step, a third of its instructions). An option of the compiler's own: one that does not
# know it builds the file without.
FILE_FLAGS = {"attention": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libtrida_hip.so)")


def _compile(src: Path) -> Path:
    obj = OBJ / (src.stem + ".o")
    extra = FILE_FLAGS.get(src.stem, [])
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    r = subprocess.run([*cmd, *extra], capture_output=True, text=True)
    if r.returncode != 0 and extra and "Unknown command line argument" in r.stderr:
        print(f"[trida] {src.name}: this compiler does not know {' '.join(extra)}; built without (slower kernels)", flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{r.stdout}\n{r.stderr}")
    return obj


def build(verbose: bool = True) -> Path:
    OBJ.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"[trida] built {LIB} from {len(sources)} sources ({ARCH})", flush=True)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
