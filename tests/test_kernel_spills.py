"""No kernel of the fused lm_head's DMA sweep stores a spilled register while lanes are switched off: such a store leaves the other lanes'
copies as they were, and a reload behind the branch reads what was never written (seen once, as wrong partials for masked batches).
The compiler decides this anew at every edit, so the built library's own code objects are read and followed on the CPU."""
import os
import re
import struct
import subprocess

import pytest

from tome_amd import build

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
KERNEL = "fused_lmhead_dma_kernel"


def code_objects(path):
    data = open(path, "rb").read()
    at = data.find(BUNDLE)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + name_len]:
                yield data[at + offset:at + offset + size]
            p += 24 + name_len
        at = data.find(BUNDLE, at + len(BUNDLE))


def kernels(listing):
    """name -> [(address, instruction, branch target or None)]"""
    found, body = {}, None
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.*)>:$", line)
        if head:
            body = found.setdefault(head.group(2), []) if KERNEL in head.group(2) else None
            start = int(head.group(1), 16)
            continue
        m = re.match(r"^\s+(\S.*?)\s*//\s*([0-9A-F]+):", line) if body is not None else None
        if m:
            to = re.search(r"<[^+>]*(?:\+0x([0-9a-f]+))?>", line.split("//", 1)[1])
            body.append((int(m.group(2), 16), m.group(1), start + int(to.group(1) or "0", 16) if to else None))
    return found


def scalar_registers(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]|s(\d+)", operand)
    if operand == "vcc":
        return ["vcc_lo", "vcc_hi"]
    if not m:
        return [operand] if operand in ("vcc_lo", "vcc_hi") else []
    return [f"s{k}" for k in range(int(m.group(1)), int(m.group(2)) + 1)] if m.group(1) else [f"s{m.group(3)}"]


class Lanes:
    """Which lanes are on: () all of them, longer tuples narrower; and which registers (and lanes of spill registers) hold such a mask."""

    def __init__(self, on=(), held=None):
        self.on, self.held = on, dict(held or {})

    def copy(self):
        return Lanes(self.on, self.held)

    def mask_in(self, operand):
        regs = scalar_registers(operand)
        tags = [self.held.get(r) for r in regs]
        return tags[0][0] if len(tags) == 2 and all(tags) and tags[0] == (tags[1][0], 0) and tags[1][1] == 1 else None

    def put(self, operand, on):
        for half, r in enumerate(scalar_registers(operand)):
            self.held[r] = (on, half)

    def step(self, where, text):
        """Runs one instruction; a fault's text, or None."""
        op, _, rest = text.partition(" ")
        args = [a.strip() for a in rest.split(",")]
        if op.startswith("scratch_store"):
            return f"{text} with lanes off" if self.on else None
        if op.startswith("s_") and "saveexec" in op:
            before, source = self.on, self.mask_in(args[1])
            if op.startswith("s_and_"):
                self.on = before + (where,)
            elif op.startswith("s_or_"):
                self.on = () if args[1] == "-1" else source if source is not None else before
            else:
                self.on = before + (where,)
            self.put(args[0], before)
        elif args[0] == "exec" or args[0].startswith("exec_"):
            if op == "s_or_b64" and args[1] == "exec":
                back = self.mask_in(args[2])
                if back is None:
                    return f"{text}: the mask is not followed"
                self.on = back
            elif op == "s_mov_b64":
                known = () if args[1] == "-1" else self.mask_in(args[1])
                self.on = known if known is not None else self.on + (where,)
            else:
                self.on = self.on + (where,)
        elif op == "s_mov_b64" and args[1] == "exec":
            self.put(args[0], self.on)
        elif op == "s_xor_b64" and [m for m in map(self.mask_in, args[1:]) if m is not None]:
            # The lanes that a branch leaves out, out of those that came to it: with them the mask is again what it was.
            self.put(args[0], [m for m in map(self.mask_in, args[1:]) if m is not None][0])
        elif op == "v_writelane_b32":
            self.move((args[0], args[2]), self.held.get(args[1]))
        elif op == "v_readlane_b32":
            self.move(args[0], self.held.get((args[1], args[2])))
        elif op in ("s_mov_b64", "s_mov_b32"):
            tags = [self.held.get(r) for r in scalar_registers(args[1])]
            for r, tag in zip(scalar_registers(args[0]), tags or [None, None]):
                self.move(r, tag)
        elif not op.startswith(("s_cmp", "s_bitcmp", "s_cbranch", "s_branch", "s_wait")):
            written = args[:2] if re.match(r"v_(mad_[ui]64|div_scale|\w+_co_)", op) else args[:1]
            for operand in written:
                for r in scalar_registers(operand):
                    self.held.pop(r, None)
        return None

    def move(self, key, tag):
        if tag is None:
            self.held.pop(key, None)
        else:
            self.held[key] = tag

    def meet(self, other):
        """What holds on both ways into a block (None: nothing new).  Where they differ in the lanes the narrower one counts."""
        on = max(self.on, other.on, key=len)
        held = {k: v for k, v in self.held.items() if other.held.get(k) == v}
        return None if on == self.on and len(held) == len(self.held) else Lanes(on, held)


def faults(body):
    index = {address: i for i, (address, _, _) in enumerate(body)}
    branch = ("s_branch", "s_cbranch")
    heads = {index[to] for _, text, to in body if to is not None and text.startswith(branch)}
    entry, work, found = {0: Lanes()}, [0], {}
    while work:
        i = work.pop()
        lanes = entry[i].copy()
        while True:
            address, text, to = body[i]
            fault = lanes.step(address, text)
            if fault:
                found[address] = fault
            after = [] if text.startswith(("s_endpgm", "s_branch")) else [i + 1]
            if to is not None and text.startswith(branch):
                after.append(index[to])
            if after == [i + 1] and i + 1 not in heads:
                i += 1
                continue
            for j in after:
                met = entry[j].meet(lanes) if j in entry else lanes.copy()
                if met:
                    entry[j] = met
                    work.append(j)
            break
    return [found[a] for a in sorted(found)]


NARROWED = ["s_and_saveexec_b64 s[2:3], vcc", "s_cbranch_execz 1 -> {after}", "v_mov_b32_e32 v1, v2"]
STORE = "scratch_store_dword off, v9, off offset:48"


@pytest.mark.parametrize("lines,wrong", [
    ([STORE], 0),
    (NARROWED + [STORE, "s_or_b64 exec, exec, s[2:3]"], 1),                                                # inside the branch
    (NARROWED + ["s_or_b64 exec, exec, s[2:3]", STORE], 0),                                                # behind it
    (NARROWED + ["v_writelane_b32 v255, s2, 4", "v_writelane_b32 v255, s3, 5", "s_mov_b32 s2, 0", "v_readlane_b32 s6, v255, 4",
                 "v_readlane_b32 s7, v255, 5", "s_or_b64 exec, exec, s[6:7]", STORE], 0),                  # the mask itself spilled
    (NARROWED + ["s_mov_b32 s2, 0", "s_or_b64 exec, exec, s[2:3]", STORE], 2),                             # the mask lost
    (["s_mov_b64 s[4:5], exec", "s_and_b64 s[0:1], s[4:5], vcc", "s_xor_b64 s[6:7], s[0:1], s[4:5]", "s_mov_b64 exec, s[0:1]", STORE,
      "s_or_b64 exec, exec, s[6:7]", STORE], 1),                                                           # the long form of the same
    (["s_or_saveexec_b64 s[2:3], -1", STORE, "s_mov_b64 exec, s[2:3]", STORE], 0),                         # all lanes on for the store
])
def test_lanes_are_followed(lines, wrong):
    after = next((i for i, x in enumerate(lines) if x.startswith(("s_or_b64 exec", "v_writelane"))), 0)
    body = [(i, x.split(" -> ")[0], after if "->" in x else None) for i, x in enumerate(lines + ["s_endpgm"])]
    assert len(faults(body)) == wrong, faults(body)


def test_no_spill_store_with_lanes_switched_off(tmp_path):
    if not os.path.exists(build.LIB_PATH):
        build.build()
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    seen, spilling = 0, 0
    for k, code in enumerate(code_objects(build.LIB_PATH)):
        if KERNEL.encode() not in code:
            continue
        path = tmp_path / f"{k}.co"
        path.write_bytes(code)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(path)], check=True, capture_output=True, text=True).stdout
        for name, body in kernels(listing).items():
            seen += 1
            spilling += any(text.startswith("scratch_store") for _, text, _ in body)
            assert faults(body) == [], name
    assert seen >= 60 and spilling > 0
