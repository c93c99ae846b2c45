"""Build libixgdn.so (HIP, gfx950) in-tree with hipcc, and _bind.so, the Python mirror's call path.

    python -m baloon_amd.build           # compile every csrc/*.hip and link the library; csrc/bind.cpp
    python baloon_amd/build.py           # the same without importing the package (and, without torch, no _bind.so)

Each translation unit is compiled for gfx950 only, with packed-FP32 instruction selection
disabled (-packed-fp32-ops), and with kernel resource-usage remarks captured to
``_build/resource_usage.txt`` (one line per kernel: ``name=... VGPRs=.. AGPRs=.. ScratchSize=..
Occupancy=.. SGPRsSpill=.. VGPRsSpill=.. LDSSize=..``) so tests can assert that no hot kernel
spills to scratch and report SGPR spills, which land in VGPR lanes (v_writelane/v_readlane).
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libixgdn.so")
BIND = os.path.join(PKG, "_bind.so")
RESOURCE_REPORT = os.path.join(BUILD, "resource_usage.txt")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", INCLUDE, "-I", CSRC,
]


# Per-file additions. The decode kernels' atomics are single-lane group counters whose
# results are used only at the end of a workgroup; the atomic optimizer would expand each
# into a wave scan that broadcasts the result right away, waiting out the atomic's round
# trip (and every load in flight) in the middle of the state stream.
FILE_FLAGS = {
    "gdn_decode.hip": ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"],
}


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> tuple[str, str]:
    obj = os.path.join(BUILD, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, *FILE_FLAGS.get(os.path.basename(src), []), "-Rpass-analysis=kernel-resource-usage",
           "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj, r.stderr


def _resource_summary(remarks: str) -> str:
    """Condense -Rpass-analysis=kernel-resource-usage remarks to one line per kernel."""
    lines, cur = [], None
    for ln in remarks.splitlines():
        m = re.search(r"remark:\s+(Function Name|VGPRs|AGPRs|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]|"
                      r"VGPRs Spill|SGPRs Spill|LDS Size \[bytes/block\]):\s*(\S+)", ln)
        if not m:
            continue
        key, val = m.group(1), m.group(2)
        if key == "Function Name":
            cur = {"name": val}
            lines.append(cur)
        elif cur is not None:
            cur[key.split(" [")[0].replace(" ", "")] = val      # e.g. "SGPRs Spill" -> SGPRsSpill
    out = []
    for d in lines:
        out.append(" ".join(f"{k}={v}" for k, v in d.items()))
    return "\n".join(out) + "\n"


def _build_bind() -> None:
    """_bind.so: host C++ against the Python and torch headers (csrc/bind.cpp)."""
    import sysconfig

    try:
        import torch
        from torch.utils.cpp_extension import include_paths
    except ImportError as e:                     # C and C++ callers need the library alone
        print(f"no Python binding: {e}")
        return

    rocm = os.path.dirname(os.path.dirname(HIPCC))
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    inc = [INCLUDE, sysconfig.get_paths()["include"], *include_paths(), os.path.join(rocm, "include")]
    tmp = BIND + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[a for p in inc for a in ("-isystem", p)], os.path.join(CSRC, "bind.cpp"), "-o", tmp,
           "-L", libs, "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"the Python binding failed to build:\n{r.stderr}")
    os.replace(tmp, BIND)


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        bind = ex.submit(_build_bind)
        results = list(ex.map(_compile, srcs))
    objs = [o for o, _ in results]
    remarks = "".join(r for _, r in results)
    with open(RESOURCE_REPORT, "w") as f:
        f.write(_resource_summary(remarks))
    tmp = LIB + ".tmp"
    r = subprocess.run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    bind.result()                                # the library stands without it
    if verbose:
        print(open(RESOURCE_REPORT).read(), end="")
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
