"""Looks through a library's gfx950 code for lane-broadcast (DPP) hazards.

A vector instruction may read a register through DPP no sooner than 2 wait
states after another vector instruction wrote it, and no sooner than 5 after one
wrote EXEC (the CDNA instruction set's table of manually inserted wait states).
The compiler keeps to that for its own instructions.  It cannot see into the
inline assembly of rowbc.h and m2lv_kernels.h, whose coefficient registers are
meant to come from loads: a register copy or a spill placed just before such a
statement would give wrong results now and then.  The build runs this after
linking and fails on any hit.

    python3 check_dpp.py LIBRARY
"""
import concurrent.futures
import os
import re
import shutil
import subprocess
import sys
import tempfile

OBJDUMP = os.environ.get("LLVM_OBJDUMP", "/opt/rocm/llvm/bin/llvm-objdump")
WAIT_VGPR, WAIT_EXEC = 2, 5
EXEC = -1

_SYMBOL = re.compile(r"^([0-9a-f]+) <(.+)>:$")
_TARGET = re.compile(r"<(.+?)(?:\+0x([0-9a-f]+))?>\s*$")
_RANGE = re.compile(r"^-?\|?v\[(\d+):(\d+)\]")
_SINGLE = re.compile(r"^-?\|?v(\d+)\b")


def _regs(operand):
    m = _RANGE.match(operand)
    if m:
        return frozenset(range(int(m.group(1)), int(m.group(2)) + 1))
    m = _SINGLE.match(operand)
    return frozenset([int(m.group(1))]) if m else frozenset()


def _written(op, args):
    """VGPRs (or EXEC) that a vector instruction writes."""
    if not op.startswith("v_") or op.startswith(("v_readlane", "v_readfirstlane", "v_nop")):
        return frozenset()
    if op.startswith("v_cmpx"):
        return frozenset([EXEC])
    if op.startswith("v_cmp"):
        return frozenset()
    if "swap" in op:  # both operands
        return _regs(args[0]) | _regs(args[1])
    return _regs(args[0]) if args else frozenset()


class Code:
    """Instructions of a disassembly, with what each can follow."""

    def __init__(self, lines):
        self.text, self.wait, self.written, self.dpp, self.ends = [], [], [], [], []
        addresses, targets, symbols = {}, [], {}
        for line in lines:
            m = _SYMBOL.match(line)
            if m:
                symbols[m.group(2)] = int(m.group(1), 16)
                continue
            body, _, comment = line.partition("//")
            words = body.split(None, 1)
            if not words or not comment:
                continue
            op, i = words[0], len(self.text)
            args = [a.strip() for a in words[1].split(",")] if len(words) > 1 else []
            addresses[int(comment.split(":", 1)[0], 16)] = i
            self.text.append(body.strip())
            self.wait.append(int(args[0], 0) + 1 if op == "s_nop" else 1)
            self.written.append(_written(op, args))
            read = frozenset()
            if op.endswith("_dpp"):  # the first vector source
                read = next((r for r in map(_regs, args[1:]) if r), frozenset())
            self.dpp.append(read)
            self.ends.append(op in ("s_branch", "s_endpgm", "s_setpc_b64", "s_trap"))
            if op.startswith(("s_branch", "s_cbranch")):
                m = _TARGET.search(comment)
                if m:
                    targets.append((i, m.group(1), int(m.group(2) or "0", 16)))
        self.jumps = {}
        for i, name, offset in targets:
            at = addresses.get(symbols.get(name, -1) + offset)
            if at is not None:
                self.jumps.setdefault(at, []).append(i)

    def _before(self, i):
        if i > 0 and not self.ends[i - 1]:
            yield i - 1
        yield from self.jumps.get(i, ())

    def _written_within(self, i, regs, states):
        for p in self._before(i):
            if self.written[p] & regs:
                return p
            if states > self.wait[p]:
                hit = self._written_within(p, regs, states - self.wait[p])
                if hit is not None:
                    return hit
        return None

    def hazards(self):
        for i, regs in enumerate(self.dpp):
            if not regs:
                continue
            hit = self._written_within(i, regs, WAIT_VGPR)
            if hit is None:
                hit = self._written_within(i, frozenset([EXEC]), WAIT_EXEC)
            if hit is not None:
                yield self.text[hit], self.text[i]


def check_object(path):
    r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", path], capture_output=True, text=True, check=True)
    code = Code(r.stdout.splitlines())
    return sum(1 for d in code.dpp if d), list(code.hazards())


def check_library(path):
    """(DPP reads, hazards as (write, read) texts) over the library's device code."""
    with tempfile.TemporaryDirectory() as tmp:
        lib = shutil.copy(path, tmp)
        subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp, check=True, stdout=subprocess.DEVNULL)
        objects = sorted(os.path.join(tmp, f) for f in os.listdir(tmp) if "amdgcn" in f)
        if not objects:
            raise RuntimeError("no device code in %s" % path)
        with concurrent.futures.ProcessPoolExecutor(min(8, os.cpu_count() or 1)) as pool:
            results = list(pool.map(check_object, objects))
    return sum(n for n, _ in results), [h for _, hs in results for h in hs]


def main(path):
    reads, hits = check_library(path)
    for write, read in hits[:20]:
        print("DPP hazard: %s  <-  %s" % (read, write))
    print("check_dpp: %d reads, %d hazards" % (reads, len(hits)))
    return 1 if hits else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1]))
