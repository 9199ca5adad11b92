"""Build-time check of the kernels' machine code (run by the Makefile after
the library links).

Disassembles the gfx950 code objects of a file built here (its .hip_fatbin
section) and fails on lane reads too close to their neighbours: the hardware
needs one wait state between a vector instruction that writes a VGPR and the
v_readfirstlane / v_readlane that reads it, and two between that lane read
and a vector instruction that reads its SGPR.  The compiler inserts them
around its own instructions, not around those of an inline asm.

usage: python3 check_code.py FILE
"""
import os
import re
import subprocess
import sys
import tempfile

LLVM = "/opt/rocm/llvm/bin"
TARGET = b"hipv4-amdgcn-amd-amdhsa--gfx950"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects in FILE's offload bundles."""
    data = open(path, "rb").read()

    def u64(at):
        return int.from_bytes(data[at:at + 8], "little")

    start = data.find(MAGIC)
    while start >= 0:
        at = start + len(MAGIC)
        count, at = u64(at), at + 8
        for _ in range(count):
            off, size, name_len = u64(at), u64(at + 8), u64(at + 16)
            if data[at + 24:at + 24 + name_len] == TARGET:
                yield data[start + off:start + off + size]
            at += 24 + name_len
        start = data.find(MAGIC, at)


def disassemble(code):
    """Lines of a code object's listing: `<kernel>:`, `<Ln>:` and instructions."""
    with tempfile.TemporaryDirectory() as d:
        co = os.path.join(d, "co")
        with open(co, "wb") as f:
            f.write(code)
        out = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn",
                              "--no-leading-addr", "--symbolize-operands", co], check=True,
                             capture_output=True, text=True).stdout
    return [line.split("//")[0].strip() for line in out.splitlines()]


def registers(text, kind):
    """The numbers of the registers of a kind ("v" or "s") in operands."""
    out = set()
    for lo, hi, one in re.findall(rf"(?<![\w]){kind}(?:\[(\d+):(\d+)\]|(\d+))(?![\w:])", text):
        out.update(range(int(lo), int(hi) + 1) if lo else [int(one)])
    return out


def wait_states(op, args):
    return int(args) + 1 if op == "s_nop" else 1


def lane_read_hazards(lines):
    """(kernel, instruction, instruction) of lane reads without their wait states."""
    found = []
    kernel = None
    recent = []  # (wait states since, VGPRs written, SGPR of a lane read, text)
    for text in lines:
        m = re.match(r"<(\w+)>:$", text)
        if m:
            if not re.match(r"L\d+$", m[1]):
                kernel = m[1]
            recent = []  # what comes before a label is not known
            continue
        if not text:
            continue
        op, _, args = text.partition(" ")
        dst, _, src = args.partition(",")
        vector = op.startswith("v_")
        lane_read = op.startswith(("v_readfirstlane", "v_readlane"))
        if vector:
            vs, ss = registers(src, "v"), registers(src, "s")
            for wait, written, sgpr, before in recent:
                if lane_read and wait < 1 and written & vs:
                    found.append((kernel, before, text))
                if wait < 2 and sgpr & ss:
                    found.append((kernel, before, text))
        gap = wait_states(op, args)
        recent = [(w + gap, *r) for w, *r in recent if w + gap < 2]
        if vector:
            recent.append((0, set() if lane_read else registers(dst, "v"),
                           registers(dst, "s") if lane_read else set(), text))
    return found


def main(argv):
    bad = []
    kernels = 0
    for code in code_objects(argv[1]):
        lines = disassemble(code)
        kernels += sum(1 for t in lines if re.match(r"<_Z\w+>:$", t))
        bad += lane_read_hazards(lines)
    for kernel, before, after in bad:
        print(f"check_code: {kernel}: `{after}` too soon after `{before}`", file=sys.stderr)
    if bad or not kernels:
        return 1
    print(f"check_code: {kernels} kernels, lane reads have their wait states")
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv))
