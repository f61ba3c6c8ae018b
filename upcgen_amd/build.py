"""Build libupcgen_amd.so (HIP kernels for gfx950 + C ABI + C++ facade) in-tree.

Usage: python -m upcgen_amd.build   (or upcgen_amd.build.build()).
       python -m upcgen_amd.build --resources [FILTER]
           the compiler's resource report of every kernel (VGPRs, AGPRs,
           SGPRs, spills, private and LDS bytes, occupancy), read from the
           metadata of a device-only compile; FILTER keeps kernels whose
           name contains it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
ROOT = os.path.dirname(HERE)
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libupcgen_amd.so")
EXE = os.path.join(HERE, "upcgen")

HIP_SOURCES = ["upc_capi.hip", "upc_tables.hip", "upc_flux_lumi.hip", "upc_flux_rows.hip", "upc_lumi.hip", "upc_xsec.hip", "upc_mfma.hip",
               "upc_surrogate.hip", "upc_events.hip", "upc_batch.hip", "upc_noalloc.hip"]
CXX_SOURCES = ["UpcCrossSection.cpp", "UpcGenerator.cpp"]

ARCH = os.environ.get("UPC_OFFLOAD_ARCH", "gfx950")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
COMMON = ["-O3", "-fPIC", "-std=c++17", f"-I{os.path.join(ROOT, 'include')}", f"-I{CSRC}"]
# Packed-FP32 VALU forms are disabled for every HIP translation unit.
HIPFLAGS = COMMON + [f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                     "-munsafe-fp-atomics", "-Wno-unused-command-line-argument"]
# The QAGS kernels run at their register budget: without this the compiler lifts
# address and constant computations out of their long loops and spills them
# (k_flux_qags_team 155 -> 122 VGPRs, k_flux_qags 157 -> 127; k_flux_qags_table 47
# -> 0 spilled for a grid's rows, 63 -> 12 for a batch's).
QAGS_FLAGS = ["-mllvm", "-disable-machine-licm"]
QAGS_SOURCES = {"upc_flux_lumi.hip", "upc_batch.hip", "upc_noalloc.hip"}


def _hip_flags(src: str) -> list:
    return HIPFLAGS + (QAGS_FLAGS if src in QAGS_SOURCES else [])


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"command failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return r


def _compile(src: str) -> str:
    path = os.path.join(CSRC, src)
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    # host-only C++ of the facade is compiled as HIP too: it calls the HIP runtime
    flags = _hip_flags(src)
    extra = ["-x", "hip"]
    _run([HIPCC] + flags + extra + ["-c", path, "-o", obj])
    return obj


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    sources = HIP_SOURCES + [s for s in CXX_SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", tmp] + objs)
    os.replace(tmp, LIB)
    main = os.path.join(CSRC, "main.cpp")
    if os.path.exists(main):
        _run([HIPCC] + HIPFLAGS + ["-x", "hip", main, "-o", EXE, f"-L{HERE}", "-lupcgen_amd",
                                   "-Wl,-rpath,$ORIGIN"])
    probe = os.path.join(ROOT, "tests", "facade_members.cpp")
    if os.path.exists(probe):  # test driver of facade members the CLI does not reach
        _run([HIPCC] + HIPFLAGS + ["-x", "hip", probe, "-o", os.path.join(ROOT, "tests", "facade_members"),
                                   f"-L{HERE}", "-lupcgen_amd", "-Wl,-rpath,$ORIGIN/../upcgen_amd"])
    if verbose:
        print(f"built {LIB}")
    return LIB


def _demangled(names):
    r = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True)
    out = r.stdout.splitlines() if r.returncode == 0 else []
    return out if len(out) == len(names) else list(names)


def resources(name_filter: str = "") -> list:
    """Per-kernel resource usage from the compiler's code-object metadata."""
    import re
    import tempfile
    rows = []
    with tempfile.TemporaryDirectory() as tmp:
        for src in HIP_SOURCES:
            asm = os.path.join(tmp, src + ".s")
            _run([HIPCC] + _hip_flags(src) + ["--cuda-device-only", "-S", "-x", "hip", os.path.join(CSRC, src), "-o", asm])
            text = open(asm).read()
            for m in re.finditer(r"\n  - \.agpr_count:(.*?)(?=\n  - \.|\n\.end_amdgpu_metadata)", text, re.S):
                block = m.group(0)

                def get(key, default=0):
                    k = re.search(r"\." + key + r":\s+(\S+)", block)
                    return k.group(1) if k else default
                rows.append({"source": src, "symbol": get("name", ""), "vgpr": int(get("vgpr_count")),
                             "agpr": int(get("agpr_count")), "sgpr": int(get("sgpr_count")),
                             "vgpr_spill": int(get("vgpr_spill_count")), "sgpr_spill": int(get("sgpr_spill_count")),
                             "private_bytes": int(get("private_segment_fixed_size")),
                             "lds_bytes": int(get("group_segment_fixed_size")),
                             "waves_per_simd_by_regs": min(8, 512 // max(1, -(-(int(get("vgpr_count")) +
                                                                            int(get("agpr_count"))) // 8) * 8))})
    for r, d in zip(rows, _demangled([r["symbol"] for r in rows])):
        r["kernel"] = d
    return [r for r in rows if name_filter in r["kernel"]]


if __name__ == "__main__":
    if len(sys.argv) > 1 and sys.argv[1] == "--resources":
        rows = resources(sys.argv[2] if len(sys.argv) > 2 else "")
        print(f"{'kernel':<78} {'vgpr':>5} {'agpr':>5} {'sgpr':>5} {'v-spill':>7} {'s-spill':>7} "
              f"{'private B':>9} {'LDS B':>7} {'waves/SIMD (regs)':>17}")
        for r in rows:
            print(f"{r['kernel'][:78]:<78} {r['vgpr']:>5} {r['agpr']:>5} {r['sgpr']:>5} {r['vgpr_spill']:>7} "
                  f"{r['sgpr_spill']:>7} {r['private_bytes']:>9} {r['lds_bytes']:>7} {r['waves_per_simd_by_regs']:>17}")
        sys.exit(0)
    build(verbose=True)
    sys.exit(0)
