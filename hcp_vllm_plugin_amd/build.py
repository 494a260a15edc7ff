"""Build ``libhcp_mi355x.so`` in-tree with hipcc for gfx950.

``python -m hcp_vllm_plugin_amd.build`` (or ``__graft_entry__.build()``).
Always recompiles; the output lands next to this file so it is found by
``hcp_vllm_plugin_amd._lib`` and travels with the source tree.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
ROOT = os.path.dirname(HERE)
OUT = os.path.join(HERE, "libhcp_mi355x.so")

# (source, extra flags) of each object: the prefill kernels once per column
# width, so that their instantiations compile side by side
OBJECTS = [
    ("attn_fwd.hip", ["-DHCP_FWD_D=128"]),
    ("attn_fwd.hip", ["-DHCP_FWD_D=256"]),
    ("attn_fwd.hip", ["-DHCP_FWD_D=64"]),
    ("decode.hip", []),
    ("abi.hip", []),
    ("merge.hip", []),
    ("cache.hip", []),
]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed-FP32 VALU forms are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results stay in arch VGPRs: the softmax reads the score tiles with
    # VALU ops, which cannot take AGPR operands
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the GPU-only feature flag; drop that noise
    err = "\n".join(ln for ln in res.stderr.splitlines() if "packed-fp32-ops" not in ln)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


def build(verbose: bool = False) -> str:
    cc = hipcc()
    with tempfile.TemporaryDirectory() as tmp, ThreadPoolExecutor(os.cpu_count() or 1) as pool:
        objs = [os.path.join(tmp, f"{i}.o") for i in range(len(OBJECTS))]
        jobs = [pool.submit(_run, [cc, *HIPCC_FLAGS, *flags, "-I", os.path.join(ROOT, "include"),
                                   "-c", os.path.join(CSRC, src), "-o", obj], verbose)
                for (src, flags), obj in zip(OBJECTS, objs)]
        for j in jobs:
            j.result()
        lib = OUT + ".tmp"
        _run([cc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs,
              "-Wl,-rpath,/opt/rocm/lib", "-o", lib], verbose)
    os.replace(lib, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
