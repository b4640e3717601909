"""Builds libmoe_gfx950.so in-tree with hipcc (gfx950 only; cross-compiles without a GPU).

    python -m iris_testing_amd.csrc.build
"""
from __future__ import annotations

import os
import re
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "libmoe_gfx950.so")
SOURCES = ["capi.hip", "route.hip", "dispatch.hip", "grouped_gemm.hip", "gemm_small.hip", "gemm_duo.hip", "step.hip", "diag.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
LLVM = os.environ.get("ROCM_LLVM", "/opt/rocm/llvm/bin")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
    # a*b+c stays two roundings unless fmaf() is written out (the combine is specified as multiply-then-add)
    "-ffp-contract=off",
    # keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(HERE, src.replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(HERE, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip() and verbose:
        print(err, file=sys.stderr)
    return obj


def disassemble(path: str) -> str:
    """The gfx950 code of an object file or library, as llvm-objdump prints it ('' if it holds none)."""
    run = lambda *cmd: subprocess.run(cmd, capture_output=True, text=True, check=True).stdout  # noqa: E731
    if ".hip_fatbin" not in run(f"{LLVM}/llvm-objdump", "-h", path):
        return ""
    text = []
    with tempfile.TemporaryDirectory() as d:
        fat, code = os.path.join(d, "fat"), os.path.join(d, "code")
        run(f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", path, os.path.join(d, "rest"))
        magic = b"__CLANG_OFFLOAD_BUNDLE__"
        for part in open(fat, "rb").read().split(magic)[1:]:  # (a library holds a bundle for each of its objects)
            with open(fat, "wb") as f:
                f.write(magic + part)
            run(f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}",
                "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={code}")
            text.append(run(f"{LLVM}/llvm-objdump", "-d", code))
    return "".join(text)


def _scalar_registers(operand: str) -> set:
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    return {int(operand[1:])} if re.fullmatch(r"s\d+", operand) else set()


WAIT_STATES = 5  # from a vector instruction's write of a scalar register to a load that takes it as base or descriptor


def early_loads(text: str):
    """(loads to LDS, those that stand fewer than WAIT_STATES wait states behind a vector instruction that wrote one of their scalar
    registers, straight on or over a branch) in llvm-objdump's text.  Such loads are written in inline assembly, and the compiler, which keeps
    its own loads apart, does not count across the start of a statement."""
    functions, seen, early = [], 0, []
    if "load_lds" not in text and not re.search(r"buffer_load\S* .* lds\b", text):
        return 0, []
    for line in text.splitlines():
        m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if m:
            functions.append((m[1], []))
        elif functions and "//" in line:
            code, at = line.split("//")[:2]
            op, *args = code.replace(",", " ").split()
            load = "load_lds" in op or (op.startswith("buffer_load") and "lds" in args)
            reads = set().union(*map(_scalar_registers, args[1:])) if load else set()
            writes = set()
            if args and not op.startswith(("s_cmp", "s_bitcmp", "s_waitcnt", "s_nop")):
                writes = _scalar_registers(args[0])
                if op.startswith("v_") and ("_co_" in op or "div_scale" in op or op.startswith("v_mad_")):  # (a carry or a flag besides)
                    writes = writes | _scalar_registers(args[1])
            to = re.search(r"\+0x([0-9a-f]+)>", at) if "branch" in op else None
            functions[-1][1].append((op, writes, int(args[0], 0) + 1 if op == "s_nop" else 1, reads, int(at.split(":")[0], 16), int(to[1], 16) if to else 0))

    def check(name, before, load):
        need, states = set(load[3]), 0
        for op, writes, n, _, _, _ in reversed(before):
            if states >= WAIT_STATES or not need:
                return
            if op.startswith("v_") and writes & need:
                early.append(f"{name}: {load[0]} at {load[4]:#x}, {states} wait states behind {op}")
                return
            if op.startswith("s_"):
                need -= writes
            states += n
    for name, ins in functions:
        start, index = ins[0][4] if ins else 0, {x[4]: i for i, x in enumerate(ins)}
        for i, x in enumerate(ins):
            if x[3]:
                seen += 1
                check(name, ins[max(0, i - 16):i], x)
            if x[0].startswith(("s_branch", "s_cbranch")) and start + x[5] in index:
                j = index[start + x[5]]
                for n in range(j, min(j + 8, len(ins))):
                    if ins[n][3]:
                        check(name, ins[max(0, i - 16):i + 1] + ins[j:n], ins[n])
    return seen, early


def build(verbose: bool = True) -> str:
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(HERE, s))]
    with ThreadPoolExecutor(max_workers=7) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    early = early_loads(disassemble(LIB))[1]
    if early:
        os.remove(LIB)
        raise RuntimeError("loads to LDS that take a scalar register too early:\n" + "\n".join(early))
    return LIB


if __name__ == "__main__":
    print(build())
