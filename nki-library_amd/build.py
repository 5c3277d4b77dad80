"""Build libmoe_gfx950.so (hand-written HIP kernels + C ABI) for gfx950 with hipcc.

Usage: ``python nki-library_amd/build.py``.  The library is written in-tree to
``nki-library_amd/nkilib/_lib/libmoe_gfx950.so`` where ``nkilib._native`` loads it.
hipcc cross-compiles, so no GPU is needed to build.  Translation units are compiled in
parallel into ``nki-library_amd/build/`` and linked; the MXFP8 large-tile GEMM
(``csrc/bwmm_mx.hip``) is compiled once per instance (``MX_INSTANCES``) plus once as the dispatcher.
"""

import os
import re
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "build")
OUT_DIR = os.path.join(HERE, "nkilib", "_lib")
OUT = os.path.join(OUT_DIR, "libmoe_gfx950.so")
SOURCES = ["rmsnorm_quant.hip", "build_blocks.hip", "combine.hip", "bwmm.hip", "bwmm_mx.hip", "bwmm_rows.hip", "router_topk.hip", "index_ops.hip", "capi.hip"]
# (stage, weight format, K that ends inside a slice) instances of the large-tile MX GEMM; formats as MX_WFMT_* in csrc/bwmm.hpp
MX_INSTANCES = [(1, 4, 0), (1, 3, 0), (1, 0, 0), (1, 1, 0), (1, 2, 0), (2, 4, 0), (2, 3, 0), (2, 0, 0), (2, 1, 0), (2, 2, 0),
                (2, 0, 1), (2, 1, 1), (2, 2, 1)]
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed fp32 ALU ops are kept off for every HIP translation unit
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# The two sources whose loads into LDS list M0 as clobbered (ld_lds_b128 in csrc/mx_tile.hpp, MXW_DMA in csrc/mx_wide.hpp,
# the like in csrc/router_topk.hip) draw one inline-asm diagnostic per such load, thousands of times; every other translation
# unit keeps the diagnostic on
MX_FLAGS = ["-Wno-inline-asm"]
M0_CLOBBER_SOURCES = ("bwmm_mx.hip", "router_topk.hip")
NOISE = "is not a recognized feature for this target"


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if NOISE not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}): {' '.join(cmd)}\n{err}")
    return err


LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


# instructions whose second operand is a scalar destination (a carry or a flag) beside the vector one
CARRY_OPS = re.compile(r"v_(\w+_co_|mad_[ui]64_|div_scale)")


def _operands(text):
    """``op a, b, c`` -> op, [a, b, c] (register ranges whole, modifiers behind an operand dropped)."""
    op, _, rest = text.partition(" ")
    return op, [o.strip().split(" ")[0] for o in re.split(r",(?![^\[]*\])", rest)] if rest else []


def _registers(operand):
    """``v7`` / ``a[0:3]`` -> (file, first, last); None for anything else."""
    m = re.fullmatch(r"([vsa])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    return m and (m[1], int(m[2] or m[3]), int(m[2] or m[4]))


def check_tile_lines(code, what):
    """What the tile loops of the large-tile GEMMs rely on and the compiler does not know of (it takes their MFMAs and loads
    for opaque statements), read from a listing of instructions:

    * it keeps nothing of its own in the accumulation registers: only MFMAs write them, and the writes of 0;
    * no vector instruction writes a scalar register within the five wait states ahead of a load that carries only the
      wait for M0 (``s_nop 0``);
    * no vector instruction but an MFMA writes an ordinary register that an MFMA within two wait states reads."""
    loads = 0
    for i, text in enumerate(code):
        op, args = _operands(text)
        if op.startswith("v_mfma"):
            reads = [r for r in map(_registers, args[1:]) if r and r[0] == "v"]
            waited, j = 0, i - 1
            while j >= 0 and waited < 2:
                before, dst = _operands(code[j])
                if before.startswith("v_") and not before.startswith("v_mfma") and dst:
                    d = _registers(dst[0])
                    if d and any(d[0] == r[0] and d[1] <= r[2] and r[1] <= d[2] for r in reads):
                        raise RuntimeError(f"{what}: {code[j]} too close to {text}")
                waited += int(dst[0], 0) + 1 if before == "s_nop" else 1
                j -= 1
        elif args and (_registers(args[0]) or "-")[0] == "a" and not (op.startswith("v_accvgpr_write") and args[1] == "0") \
                and not op.startswith(("buffer_store", "global_store", "scratch_store")):
            raise RuntimeError(f"{what}: the compiler uses an accumulation register: {text}")
        if op.startswith("buffer_load") and text.endswith("lds") and i and code[i - 1] == "s_nop 0":
            loads += 1
            for u in code[max(0, i - 7):i]:
                if u.startswith(("v_readlane", "v_readfirstlane", "v_cmp")) or CARRY_OPS.match(u):
                    raise RuntimeError(f"{what}: {u} too close to a load of the K loop")
    if loads == 0:
        raise RuntimeError(f"{what}: no K loop found in the compiled code")


def check_tile_code(obj):
    """``check_tile_lines`` of an object file (of this build's own), where the tools that list one are installed."""
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    missing = [t for t in tools if not os.path.exists(t)]
    if missing:
        return f"{obj}: its compiled code was not checked, {', '.join(missing)} not found"
    with tempfile.TemporaryDirectory() as tmp:
        fat, co = os.path.join(tmp, "fat"), os.path.join(tmp, "co")
        _run([tools[0], f"--dump-section=.hip_fatbin={fat}", obj, os.path.join(tmp, "o")])
        _run([tools[1], "--unbundle", "--type=o", f"--input={fat}", f"--output={co}",
              "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
        dis = subprocess.run([tools[2], "-d", "--no-show-raw-insn", "--no-leading-addr", co],
                             capture_output=True, text=True, check=True).stdout
    check_tile_lines([t for t in (line.split("//")[0].strip() for line in dis.splitlines()) if t], obj)
    return ""


def build(verbose=True, jobs=None):
    os.makedirs(OUT_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)
    inc = ["-I", os.path.join(ROOT, "include"), "-I", CSRC]
    units = []  # (object path, extra defines, source); the long-running instances of the large-tile GEMM go first
    for stage, fmt, ktail in MX_INSTANCES:
        units.append((os.path.join(OBJ_DIR, f"bwmm_mx_s{stage}_f{fmt}_t{ktail}.o"),
                      [*MX_FLAGS, f"-DMX_INST_STAGE={stage}", f"-DMX_INST_WFMT={fmt}", f"-DMX_INST_KTAIL={ktail}"],
                      os.path.join(CSRC, "bwmm_mx.hip")))
    for s in SOURCES:
        units.append((os.path.join(OBJ_DIR, s.replace(".hip", ".o")), MX_FLAGS if s in M0_CLOBBER_SOURCES else [],
                      os.path.join(CSRC, s)))
    cmds = [["hipcc", *FLAGS, *defs, *inc, "-c", src, "-o", obj] for obj, defs, src in units]
    if verbose:
        for c in cmds:
            print(" ".join(c), flush=True)
    jobs = jobs or min(len(cmds), os.cpu_count() or 4, 16)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        errs = list(ex.map(_run, cmds))
        errs += ex.map(check_tile_code, [u[0] for u in units[:len(MX_INSTANCES)]])
    link = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", *[u[0] for u in units], "-o", OUT]
    if verbose:
        print(" ".join(link), flush=True)
    errs.append(_run(link))
    if verbose:
        for e in errs:
            if e.strip():
                print(e)
    return OUT


if __name__ == "__main__":
    build()
    print("built", OUT)
    sys.exit(0)
