"""Build the HIP library ``miniserve_amd/libminiserve_amd.so`` for gfx950 with hipcc.

    python -m miniserve_amd.build          # or __graft_entry__.build()

Each ``csrc/*.hip`` file compiles to an object under ``miniserve_amd/_build/`` (in parallel), then
hipcc links the shared library in-tree so it travels with the source tree. Packed-FP32 VALU
instructions are disabled (``-packed-fp32-ops``) for every HIP translation unit. The host-side
CPython extension ``miniserve_amd/_hostprep`` (``csrc/hostprep.c``: packing a captured decode
step's inputs) is compiled with the system C compiler beside it.
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
LIB = PKG / "libminiserve_amd.so"
SOURCES = ["errors.hip", "quant.hip", "gemm_skinny.hip", "gemm_int8.hip", "gemm_big.hip", "gemv_rows.hip", "gemv_dec.hip", "gemv_stream.hip", "gemv_wide.hip", "norm_rope.hip", "attention.hip", "sampler.hip"]
ARCH = os.environ.get("MSA_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{ROOT / 'include'}",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found: the HIP library cannot be built")
    return path


# Per-file extra flags: keep MFMA accumulators in ordinary VGPRs. attention.hip: the prefill
# kernel rescales its output accumulators between MFMAs every key tile, and in accumulation
# registers each rescale costs a copy out and a copy back. gemm_int8.hip: in accumulation
# registers the GEMM's main loop spends 48 VALU copies per two K steps shuffling accumulators.
_VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
# attention.hip also without NaN semantics: its softmax maxima then skip the canonicalizing
# v_max_f32 x, x that IEEE mode puts before each maximum of MFMA results (the 1984-token prefill
# chunk 41.9 -> 40.7 us). The kernels compare against -inf, never against NaN.
EXTRA_FLAGS = {"attention.hip": [*_VGPR_FORM, "-fno-honor-nans"], "gemm_int8.hip": _VGPR_FORM}


def _compile(src: str) -> Path:
    obj = BUILD / (Path(src).stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, *EXTRA_FLAGS.get(src, []), "-c", str(CSRC / src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stderr[-6000:]}")
    return obj


HOSTPREP = PKG / ("_hostprep" + sysconfig.get_config_var("EXT_SUFFIX"))


def build_hostprep() -> Path:
    """Compile the CPython extension ``_hostprep`` from ``csrc/hostprep.c`` in-tree."""
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        raise RuntimeError("no C compiler found: the host extension cannot be built")
    tmp = HOSTPREP.with_suffix(".so.tmp")
    cmd = [cc, "-O2", "-fPIC", "-shared", "-Wall", "-Werror", f"-I{sysconfig.get_paths()['include']}",
           str(CSRC / "hostprep.c"), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"building _hostprep failed:\n{res.stderr[-6000:]}")
    os.replace(tmp, HOSTPREP)
    return HOSTPREP


def build(jobs: int | None = None) -> Path:
    """Compile every HIP source and link the shared library (and the host extension); returns the
    library's path."""
    BUILD.mkdir(exist_ok=True)
    jobs = jobs or min(len(SOURCES), int(os.environ.get("MAX_JOBS", "8")))
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(_compile, SOURCES))
        host = pool.submit(build_hostprep)
        host.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc link failed:\n{res.stderr[-6000:]}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(), file=sys.stderr)
