"""What csrc/gemm_wide.h relies on and no compiler checks, read from the assembly of what was just built.

Its matrix instructions are in inline asm, so that their sums stay in place; the compiler does not know how long
they take. So a kernel with them must not move a sum within a loop, read one too early after the last
instruction, or write an operand right ahead of the instruction that reads it; and a spilled register is either of these.
build.py refuses a library whose kernels do.
"""

from __future__ import annotations

import os
import re
import subprocess
import tempfile

KERNELS = re.compile(r"(gemm|moe)_wide_kernel")  # by name
OBJECTS = ("gemm_hip.cuda.o", "moe_hip.cuda.o")
SLOTS_TO_A_SUM = 18  # issue slots until a sum of 16 x 16 x 32 can be read, the longest that is documented
SLOTS_TO_AN_OPERAND = 2

_REGISTER = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)")
_LINE = re.compile(r"^\s+(\S.*?)\s*//\s*([0-9A-Fa-f]+):")


def _registers(text: str) -> set:
    found = set()
    for kind, first, last, one in _REGISTER.findall(text):
        found.update((kind, i) for i in range(int(first or one), int(last or one) + 1))
    return found


def _slots(op: str) -> int:
    return int(op.split()[1], 0) + 1 if op.startswith("s_nop") else 1


def faults(listing: str, loops: int = 1) -> list:
    """What is wrong with a kernel, given its disassembly; at least `loops` of its loops have matrix instructions."""
    ops, at = [], {}
    for line in listing.splitlines():
        m = _LINE.match(line)
        if m:
            at[int(m[2], 16)] = len(ops)
            ops.append((int(m[2], 16), m[1]))
    found, seen = [], 0
    matrix = [op.startswith("v_mfma") for _, op in ops]
    target = [_registers(op.split(",")[0]) for _, op in ops]
    used = [_registers(op) for _, op in ops]
    # loops: a branch to where matrix instructions lie ahead of it
    for i, (address, op) in enumerate(ops):
        if not op.startswith(("s_cbranch", "s_branch")):
            continue
        way = int(op.split()[1], 0)
        way -= 65536 if way > 32767 else 0
        start = at.get(address + 4 + 4 * way, i)
        inside = [j for j in range(start, i) if matrix[j]]
        if not inside:
            continue
        seen += 1
        sums = set().union(*(target[j] for j in inside))
        found += [f"a sum is moved in a loop: {ops[j][1]}" for j in range(start, i) if not matrix[j] and used[j] & sums]
    for i in range(len(ops)):
        if not matrix[i]:
            continue
        slots, j = 0, i + 1
        while j < len(ops) and slots < SLOTS_TO_A_SUM:
            if not matrix[j] and used[j] & target[i]:
                found.append(f"a sum is read or written too early: {ops[j][1]}")
            slots, j = slots + _slots(ops[j][1]), j + 1
        operands = _registers(ops[i][1].split(",", 1)[1])
        slots, j = 0, i - 1
        while j >= 0 and slots < SLOTS_TO_AN_OPERAND:
            if ops[j][1].startswith("v_") and not matrix[j] and target[j] & operands:
                found.append(f"an operand is written too late: {ops[j][1]}")
            slots, j = slots + _slots(ops[j][1]), j - 1
    if seen < loops:
        found.append(f"{seen} loops with matrix instructions where {loops} are expected")
    return found


def _run(tool: str, *args: str) -> str:
    root = os.environ.get("ROCM_PATH", "/opt/rocm")
    return subprocess.run([os.path.join(root, "llvm", "bin", tool), *args], check=True, capture_output=True, text=True).stdout


def check(folder: str) -> int:
    """Looks at the objects of a build folder. How many kernels there were; raises if one is at fault."""
    kernels = 0
    for name in OBJECTS:
        path = os.path.join(folder, name)
        if not os.path.exists(path):
            continue
        with tempfile.TemporaryDirectory() as tmp:
            bundle, code = os.path.join(tmp, "bundle"), os.path.join(tmp, "code")
            _run("llvm-objcopy", f"--dump-section=.hip_fatbin={bundle}", path, os.devnull)
            _run("clang-offload-bundler", "--unbundle", "--type=o", f"--input={bundle}",
                 "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={code}")
            notes = _run("llvm-readelf", "--notes", code)
            # a kernel's entries lie on both sides of its name, which ends with its last ones
            for entry in re.split(r"\n(?=  - \.agpr_count:)", notes):
                kernel = re.search(r"\.name:\s+(\S*)", "\n".join(l for l in entry.splitlines() if l.startswith("    .name")))
                if kernel is None or not KERNELS.search(kernel[1]):
                    continue
                kernels += 1
                for what in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"):
                    if re.search(rf"\.{what}:\s+0\b", entry) is None:
                        raise RuntimeError(f"{kernel[1]}: {what} is not 0")
            for function in re.split(r"\n(?=[0-9a-f]+ <)", _run("llvm-objdump", "-d", "--no-show-raw-insn", code)):
                title = function.split("\n", 1)[0]
                if KERNELS.search(title):
                    loops = (4 if "ILb1E" in title else 8) if "moe" in title else 1  # 1 to 4 or 8 tiles a group
                    wrong = faults(function, loops)
                    if wrong:
                        raise RuntimeError(f"{title}: {len(wrong)} faults, the first: {wrong[0]}")
    return kernels
