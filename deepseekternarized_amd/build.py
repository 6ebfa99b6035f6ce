"""Builds libbp_ternary_hip.so (the gfx950 kernels and their C ABI) in-tree with hipcc.

    python -m deepseekternarized_amd.build [--incremental]

The shared object lands next to this file; it is what ``deepseekternarized_amd.kernels.ternary_hip``
loads with ctypes. hipcc cross-compiles for gfx950 without a GPU present.
"""

from __future__ import annotations

import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB = HERE / "libbp_ternary_hip.so"
SOURCES = ["bp_api.hip", "bp_general.hip", "bp_repack.hip", "bp_route.hip", "bp_gguf.hip", "bp_huffman.hip", "bp_moe.hip", "bp_mfma.hip", "bp_mfma_tq2.hip", "bp_gemm_tq2.hip", "bp_gemm_tq2f.hip", "bp_gemm_f4.hip", "bp_mfma_tq1.hip", "bp_gemm_tq1.hip", "bp_tq1_gemv.hip", "bp_tq1_gemv_fp4.hip", "bp_tq1_gemv_cw.hip", "bp_tq2_gemv_fp4.hip"]
# Compiled twice, for launches that add to their outputs and for those that replace them (BP_REPLACES in bp_common.h).
TWICE = {"bp_mfma_tq2.hip", "bp_gemm_tq2.hip", "bp_mfma_tq1.hip", "bp_gemm_tq1.hip", "bp_tq1_gemv_fp4.hip", "bp_tq1_gemv_cw.hip", "bp_tq2_gemv_fp4.hip"}
# packed FP32 VALU ops are disabled for every device object of this library
FLAGS = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-Wall", "-Wno-unused-function", "-Wno-int-to-pointer-cast",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


# These kernels address LDS absolutely (their dynamic allocation must start at LDS address 0): a kernel of theirs
# with static LDS - e.g. a register array the compiler moved there because it was indexed dynamically - would
# compute on the wrong bytes, so the build refuses it.
NO_STATIC_LDS = {"bp_mfma_tq2.hip", "bp_gemm_tq2.hip", "bp_gemm_tq2f.hip", "bp_gemm_f4.hip", "bp_mfma_tq1.hip", "bp_gemm_tq1.hip", "bp_tq1_gemv.hip", "bp_tq1_gemv_fp4.hip", "bp_tq1_gemv_cw.hip", "bp_tq2_gemv_fp4.hip"}
_REMARK = "[-Rpass-analysis=kernel-resource-usage]"


def _units() -> list[tuple[str, str]]:
    """(source, case) of every object, the ones that take longest first; the case is "" or, of a source in TWICE, "add" or "set"."""
    units = [(s, c) for s in SOURCES for c in (("add", "set") if s in TWICE else ("",))]
    return sorted(units, key=lambda u: u[0] not in ("bp_tq1_gemv_cw.hip", "bp_tq1_gemv_fp4.hip"))


def _object(unit: tuple[str, str]) -> Path:
    return CSRC / (unit[0] + ("." + unit[1] if unit[1] else "") + ".o")


def _compile(unit: tuple[str, str]) -> Path:
    src, case = unit
    obj = _object(unit)
    check = src in NO_STATIC_LDS
    cmd = ["hipcc", *FLAGS, *([f"-DBP_REPLACES={int(case == 'set')}"] if case else []), *(["-Rpass-analysis=kernel-resource-usage"] if check else []), "-c", str(CSRC / src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    lines = [l for l in res.stderr.splitlines() if noise not in l]
    if check:  # drop the resource remarks (and the source excerpts printed under them) after reading the LDS sizes
        kept, name, skip = [], "?", 0
        for l in lines:
            if _REMARK in l:
                if "Function Name:" in l:
                    name = l.split("Function Name:")[1].split()[0]
                if "LDS Size [bytes/block]:" in l and int(l.split("LDS Size [bytes/block]:")[1].split()[0]) != 0:
                    raise RuntimeError(f"{src}: kernel {name} uses static LDS; these kernels address LDS absolutely")
                skip = 2
            elif skip and (l.lstrip().startswith("|") or l.lstrip()[:1].isdigit()):
                skip -= 1
            else:
                kept.append(l)
        lines = kept
    err = "\n".join(lines)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def _fresh(unit: tuple[str, str]) -> bool:
    """The unit's object is newer than its source and every header (used by --incremental only)."""
    obj = _object(unit)
    if not obj.exists():
        return False
    deps = [CSRC / unit[0], *CSRC.glob("*.h"), HERE.parent / "include" / "bp_ternary.h", Path(__file__)]
    return all(obj.stat().st_mtime > d.stat().st_mtime for d in deps)


def build(verbose: bool = True, incremental: bool = False) -> Path:
    """Compiles every source (``incremental``: only those older than their inputs) and links the library."""
    todo = [u for u in _units() if not (incremental and _fresh(u))]
    with ThreadPoolExecutor(max_workers=7) as pool:
        list(pool.map(_compile, todo))
    objs = [_object(u) for u in _units()]
    cmd = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,--no-undefined", *map(str, objs), "-o", str(LIB)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(incremental="--incremental" in sys.argv[1:])
