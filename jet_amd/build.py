"""Build recipe of libjet_hip.so (gfx950) -- in-tree, no JIT cache.

    python -m jet_amd.build            # compile jet_amd/_lib/libjet_hip.so

Every source under jet_amd/csrc is compiled by hipcc for gfx950 (object
files in jet_amd/_build) and linked into jet_amd/_lib/libjet_hip.so, which is
what jet_amd._native loads.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "_lib")
LIB = os.path.join(LIBDIR, "libjet_hip.so")

SOURCES = [
    "permute.hip",
    "gemm.hip",
    "gemm_f32x6.hip",
    "gemm_f64.hip",
    "misc.hip",
    "stream.hip",
    "profiler.hip",
    "network.hip",
    "jet_hip_api.hip",
    "permute_plan.cpp",
    "contract_plan.cpp",
    "network_plan.cpp",
    "tuning.cpp",
]

# The autotuned GEMM kernel table (jet_amd/autotune.py), compiled in.
TUNING_JSON = os.path.join(HERE, "data", "gemm_tuning_gfx950.json")
TUNING_INC = os.path.join(BUILD, "tuning_table.inc")

ARCH = os.environ.get("JET_HIP_ARCH", "gfx950")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-I" + os.path.join(ROOT, "include"),
    "-I" + BUILD,
    # Packed FP32 VALU instructions stay disabled on this target.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(src: str) -> str:
    path = os.path.join(CSRC, src)
    obj = os.path.join(BUILD, src + ".o")
    lang = ["-x", "hip"] if src.endswith(".hip") else []
    cmd = [HIPCC] + COMMON_FLAGS + lang + ["-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
    return obj


def write_tuning_table() -> int:
    """tuning_table.inc from the committed table: one C initializer row
    {mode, log2 M, log2 N, log2 K, log2 batch, kernel, variant} per entry and
    an end marker row; returns the number of entries."""
    import json
    rows = []
    if os.path.exists(TUNING_JSON):
        with open(TUNING_JSON) as f:
            doc = json.load(f)
        for e in doc["entries"]:
            vals = [int(x) for x in e[:7]]
            rows.append("{" + ", ".join(str(v) for v in vals) + "},")
    rows.append("{-1, 0, 0, 0, 0, 0, 0},")
    text = "// generated by jet_amd/build.py from jet_amd/data/gemm_tuning_gfx950.json\n" + \
        "\n".join(rows) + "\n"
    old = open(TUNING_INC).read() if os.path.exists(TUNING_INC) else None
    if old != text:
        with open(TUNING_INC, "w") as f:
            f.write(text)
    return len(rows) - 1


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    n_tuned = write_tuning_table()
    if verbose:
        print(f"tuning table: {n_tuned} entries")
    sources = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
