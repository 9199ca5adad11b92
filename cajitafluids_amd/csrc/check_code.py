"""Build-time check of the kernels' machine code (run by the Makefile after
the library links).

Disassembles the gfx950 code objects of a file built here (its .hip_fatbin
section) and fails on

- lane reads too close to their neighbours: the hardware needs one wait state
  between a vector instruction that writes a VGPR and the v_readfirstlane /
  v_readlane that reads it, and two between that lane read and a vector
  instruction that reads its SGPR.  The compiler inserts them around its own
  instructions, not around those of an inline asm.
- register moves before a join's lanes are back: where lanes that took a
  branch meet those that skipped it, the block opens with `s_or_b64 exec,
  exec, ...`.  Under register pressure the compiler has split a value's
  register there and put the copy (or a reload from scratch) ahead of that
  instruction, so that the lanes that skipped the branch kept garbage in the
  new register; as an index it was a wild address.

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


def early_moves(lines):
    """(kernel, label, move) of vector moves and reloads ahead of a join's exec."""
    found = []
    kernel = label = None
    moves = None  # since the label, while it may still open a join
    for text in lines:
        m = re.match(r"<(\w+)>:$", text)
        if m:
            if re.match(r"L\d+$", m[1]):
                label, moves = m[1], []
            else:
                kernel, moves = m[1], None
            continue
        if moves is None or not text:
            continue
        if re.match(r"s_or_b64 exec, exec, ", text):
            found += [(kernel, label, t) for t in moves]
            moves = None
        elif re.match(r"v_mov_b(32|64)\w* |v_accvgpr_|v_pk_mov_|scratch_load_", text):
            moves.append(text)
        elif not re.match(r"s_(?!cbranch|branch|endpgm|setpc|swappc)|v_readlane_|v_writelane_",
                          text):
            moves = None  # the block's own work: no join opens here
    return found


def main(argv):
    bad = []
    kernels = 0
    for code in code_objects(argv[1]):
        lines = disassemble(code)
        kernels += sum(1 for t in lines if re.match(r"<_Z\w+>:$", t))
        bad += [f"{k}: `{after}` too soon after `{before}`"
                for k, before, after in lane_read_hazards(lines)]
        bad += [f"{k}: `{move}` before the lanes are back at {label}"
                for k, label, move in early_moves(lines)]
    for text in bad:
        print(f"check_code: {text}", file=sys.stderr)
    if bad or not kernels:
        return 1
    print(f"check_code: {kernels} kernels, lane reads and joins in order")
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv))
