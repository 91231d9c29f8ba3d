"""Checks of the gfx950 code that mbsolve_amd.build made.

The FP64 multiply-adds with a DPP operand (row_consts in csrc/mbh_device.hpp)
are inline assembly, which the compiler's hazard handling leaves out: the
hardware does not interlock a DPP read of a register that a vector instruction
wrote in one of the two wait states before.  Nothing in the kernels writes
those registers so late, but a copy or a spill made by the register allocator
would, and the results would be wrong without an error.  ``hazards`` finds
such a sequence in the code itself; ``mbsolve_amd.build`` refuses a library
that holds one, whatever compiler and flags made it.

``resources`` gives the registers, scratch and spills of every kernel.
"""
import os
import re
import struct
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

LLVM = os.environ.get("MBSOLVE_LLVM_BIN", "/opt/rocm/llvm/bin")
CHECKED = "v_fmac_f64_dpp"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

# wait states that must lie between an instruction of the kind and a read
# through DPP (dpp) or by any operand (any)
VALU_DPP = 2
EXEC_DPP = 5
TRANS_ANY = 1
MFMA_ANY = 20
TRANS = re.compile(r"v_(rcp|rsq|sqrt|exp|log|sin|cos)_")


def code_objects(path):
    """gfx950 code objects of a shared library or object file."""
    data = open(path, "rb").read()
    out = []
    at = data.find(MAGIC)
    while at >= 0:
        count = struct.unpack_from("<Q", data, at + 24)[0]
        p = at + 32
        for _ in range(count if count < 64 else 0):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24:p + 24 + n]:
                out.append(data[at + off:at + off + size])
            p += 24 + n
        at = data.find(MAGIC, at + 24)
    return out


def _llvm(tool, args, code):
    with tempfile.NamedTemporaryFile(suffix=".elf") as f:
        f.write(code)
        f.flush()
        return subprocess.run([os.path.join(LLVM, tool)] + args + [f.name],
                              check=True, stdout=subprocess.PIPE,
                              text=True).stdout


def disassemble(code):
    return _llvm("llvm-objdump", ["-d", "--no-show-raw-insn"], code)


_REG = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _regs(text):
    out = set()
    for a, b, c in _REG.findall(text):
        out.update(range(int(a), int(b) + 1) if a else (int(c),))
    return out


class _Insn:
    __slots__ = ("addr", "op", "args", "text", "fn", "entry", "states")

    def __init__(self, addr, op, rest, fn, entry):
        self.addr, self.op, self.fn, self.entry = addr, op, fn, entry
        self.args = [a.strip() for a in rest.split(",")] if rest else []
        self.text = op + " " + rest
        self.states = int(self.args[0], 0) + 1 if op == "s_nop" else 1

    def writes(self):
        """vector registers this vector instruction writes"""
        if not self.op.startswith("v_") or not self.args:
            return set()
        n = 2 if self.op.startswith("v_swap") else 1
        return _regs(" ".join(self.args[:n]))


def _parse(listing):
    """instructions of the functions that hold a checked one"""
    insns = []
    parts = re.split(r"(?m)^[0-9a-f]+ <(.*)>:\n", listing)
    for fn, body in zip(parts[1::2], parts[2::2]):
        entry = True
        for line in body.splitlines() if CHECKED in body else ():
            m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-Fa-f]+):", line)
            if m:
                insns.append(_Insn(int(m.group(3), 16), m.group(1),
                                   m.group(2), fn, entry))
                entry = False
    return insns


def hazards(listing):
    """(number of checked instructions, list of findings) of a disassembly.

    Walks back from each checked instruction over every path that leads to
    it (branches included), as far as the longest rule reaches."""
    insns = _parse(listing)
    index = {i.addr: k for k, i in enumerate(insns)}
    preds = [[] for _ in insns]
    for k, i in enumerate(insns):
        if k + 1 < len(insns) and not insns[k + 1].entry and \
                i.op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
            preds[k + 1].append(k)
        if i.op == "s_branch" or i.op.startswith("s_cbranch"):
            d = int(i.args[0].split()[0], 0)
            to = i.addr + 4 + 4 * (d - 65536 if d >= 32768 else d)
            if to in index:
                preds[index[to]].append(k)
    found, count = [], 0
    for k, i in enumerate(insns):
        if i.op != CHECKED:
            continue
        count += 1
        dpp = _regs(i.args[1])
        used = _regs(" ".join(i.args[:3]))
        seen = {k: 0}
        todo = [k]
        while todo:
            at = todo.pop()
            dist = seen[at]
            if insns[at].entry and dist < EXEC_DPP and \
                    "kernel" not in insns[at].fn:
                found.append((i, "the caller of %s" % insns[at].fn))
            for b in preds[at]:
                j = insns[b]
                why = None
                if j.op in ("s_swappc_b64", "s_call_b64") and \
                        dist < EXEC_DPP:
                    why = "a call"
                elif j.op.startswith("v_cmpx") and dist < EXEC_DPP:
                    why = "a vector write of EXEC"
                elif ("mfma" in j.op or "smfmac" in j.op) and \
                        dist < MFMA_ANY and j.writes() & used:
                    why = "a matrix instruction"
                elif TRANS.match(j.op) and dist < TRANS_ANY and \
                        j.writes() & used:
                    why = "a transcendental"
                elif dist < VALU_DPP and j.writes() & dpp:
                    why = "a vector write of the DPP operand"
                if why:
                    found.append((i, "%s: %s" % (why, j.text)))
                d = dist + j.states
                if d < MFMA_ANY and (b not in seen or d < seen[b]):
                    seen[b] = d
                    todo.append(b)
    return count, ["%s at %x in %s after %s" % (i.text, i.addr, i.fn, why)
                   for i, why in found]


def check(path):
    """Raises if the library's code holds a hazard; returns the number of
    instructions checked."""
    total = 0
    with ThreadPoolExecutor(max_workers=6) as ex:
        listings = list(ex.map(disassemble, code_objects(path)))
    for listing in listings:
        count, found = hazards(listing)
        total += count
        if found:
            raise RuntimeError(
                "%s: %d DPP reads too early, first: %s" %
                (path, len(found), found[0]))
    return total


def resources(path):
    """{mangled kernel name: {"vgpr", "agpr", "sgpr", "lds", "vgpr_spills",
    "scratch"}}"""
    keys = {".agpr_count": "agpr", ".vgpr_count": "vgpr",
            ".sgpr_count": "sgpr", ".group_segment_fixed_size": "lds",
            ".vgpr_spill_count": "vgpr_spills",
            ".private_segment_fixed_size": "scratch"}
    out = {}
    for code in code_objects(path):
        notes = _llvm("llvm-readelf", ["--notes"], code)
        for block in re.split(r"\n  - (?=\.)", notes)[1:]:
            kv = dict(re.findall(r"(?m)^ *(\.\w+): +(\S+)$", block))
            if ".symbol" in kv:
                out[kv[".symbol"][:-3]] = {
                    name: int(kv.get(k, 0)) for k, name in keys.items()}
    return out
