"""Build the gfx950 HIP library ``edifice_amd/lib/libedifice_hip.so`` in-tree.

Every ``csrc/*.hip`` and ``csrc/*.cpp`` is compiled with hipcc for gfx950 only and
linked into one shared library exporting the C ABI declared in
``include/edifice_hip.h``.  The build always recompiles (it is also the
"does it build" check); objects go to ``edifice_amd/lib/obj``.

Packed-FP32 instructions are disabled in device code (``-packed-fp32-ops``);
hipcc's host pass warns that it does not know the feature, which is harmless.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
OBJDIR = os.path.join(LIBDIR, "obj")
LIBNAME = "libedifice_hip.so"
ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{os.path.join(os.path.dirname(HERE), 'include')}",
]


def lib_path() -> str:
    return os.path.join(LIBDIR, LIBNAME)


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


# Per-source flags.  The flash-attention backward kernels run one wave per SIMD with more
# live values than the 256 architectural VGPRs; by default the compiler then keeps MFMA
# accumulators in AGPRs and moves them back and forth around every softmax step (about 40%
# of the dQ kernel's VALU instructions).  The VGPR form of the MFMAs removes those moves
# without spilling (measured: backward 3.01 -> 2.82 ms at config 4, identical results).
# The chunked delta rule's kernels scale and convert their MFMA accumulators with VALU
# work after every product; kept in VGPRs they need no v_accvgpr moves (config 3: output
# kernel 84.6 -> 79.2 us, the others unchanged; identical results).  The row scans do the same
# with theirs at every step of a chunk (without the flag 8x2048x8x128 bf16 608 -> 623 us, KDA
# 4x1000x8x128 344 -> 350, 2x777x8x64 float32 gated 239 -> 267).
PER_FILE_FLAGS = {
    "flash_attn_bwd.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "delta_rule_chunk.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "delta_rule_row.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "delta_rule_row_bwd.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, *PER_FILE_FLAGS.get(os.path.basename(src), []), "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    noise = [ln for ln in res.stderr.splitlines() if "packed-fp32-ops" not in ln and ln.strip()]
    if noise:
        sys.stderr.write("\n".join(noise) + "\n")
    return obj


def build(jobs: int | None = None, verbose: bool = False) -> str:
    """Compile all sources for gfx950 and link the shared library; returns its path."""
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), int(os.environ.get("MAX_JOBS", "8")))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, srcs))
    out = lib_path()
    tmp = out + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, out)
    if verbose:
        print(f"built {out}")
    return out


if __name__ == "__main__":
    build(verbose=True)
