"""Ahead-of-time build of the gfx950 C-ABI library ``libdsa_mi355x.so``.

Every ``csrc/*.hip`` file is compiled with ``hipcc --offload-arch=gfx950`` and
linked into one shared library next to this file, where ``_native`` loads it.
Run ``python -m ascendc_kernel_amd.build`` (or ``__graft_entry__.build()``).
The library is rebuilt on every call; objects go to ``_build/`` at the repo root.
"""
from __future__ import annotations

import concurrent.futures as _cf
import os
import shutil
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
REPO = os.path.dirname(PKG_DIR)
LIB_NAME = "libdsa_mi355x.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
FASTCALL_PATH = os.path.join(PKG_DIR, "_fastcall.so")
ARCH = "gfx950"

# -ffp-contract=off: every fused multiply-add in the kernels is written out
# explicitly, so the rounding of each operation is the one in the source.
# The packed-fp32 feature is switched off for all device code.
HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# Per-file additions. indexer.hip: keep MFMA accumulators in VGPRs (the compiler
# otherwise places the score kernel's accumulator in AGPRs and copies it out with
# 16 v_accvgpr_read per tile; measured ~2 % faster, identical results).
EXTRA_FLAGS = {
    "indexer.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the gfx950 library cannot be built")


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str, obj: str) -> None:
    cmd = [hipcc(), *HIPCC_FLAGS, *EXTRA_FLAGS.get(os.path.basename(src), []), "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in (r.stderr or "").splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {os.path.basename(src)}:\n{err}")


def _build_fastcall() -> None:
    """``_fastcall.so``, the host-only extension of the modules' repeated calls (torch's headers)."""
    import sysconfig

    import torch
    base = os.path.dirname(torch.__file__)
    tmp = FASTCALL_PATH + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           *(f"-I{d}" for d in (f"{base}/include", f"{base}/include/torch/csrc/api/include",
                                sysconfig.get_paths()["include"], "/opt/rocm/include")),
           "-o", tmp, os.path.join(CSRC, "fastcall.cpp"), f"-L{base}/lib",
           "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for fastcall.cpp:\n{r.stderr}")
    os.replace(tmp, FASTCALL_PATH)


def build(verbose: bool = False) -> str:
    """Compile all kernels for gfx950 and link ``libdsa_mi355x.so`` (its path is returned), and
    compile the ``_fastcall`` extension."""
    objdir = os.path.join(REPO, "_build", "dsa")
    os.makedirs(objdir, exist_ok=True)
    srcs = sources()
    objs = [os.path.join(objdir, os.path.basename(s)[:-4] + ".o") for s in srcs]
    with _cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        fast = ex.submit(_build_fastcall)
        list(ex.map(_compile, srcs, objs))
        # Linked before the extension is waited for: the library is complete without it.
        tmp = LIB_PATH + ".tmp"
        cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stderr}")
        os.replace(tmp, LIB_PATH)
        fast.result()
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
