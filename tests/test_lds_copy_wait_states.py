"""The copies from memory to LDS are written by hand, where the compiler adds no wait states.  CDNA's tables of manually
inserted wait states ask for one between a write of m0 and a copy to LDS, and for five between a vector instruction's write of
a scalar register and a memory instruction that reads it.  Read from the built kernels, over every way into each copy."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from turbogpt_amd import build

LIBRARY = Path(__file__).resolve().parent.parent / "turbogpt_amd" / "libturbogpt.so"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):(?:.*<(.+?)(?:\+0x([0-9a-f]+))?>)?")


def registers_named(text):
    """Numbers of the scalar registers in an operand list; vcc and m0 by their names."""
    found = {int(n) for n in re.findall(r"\bs(\d+)\b", text)}
    for low, high in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        found.update(range(int(low), int(high) + 1))
    return found | {name for name in ("vcc", "m0") if name in text}


def written_by_vector(name, operands):
    if not name.startswith("v_"):
        return set()
    parts = operands.split(", ")
    written = registers_named(parts[0])
    if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_mad_[iu]64|v_div_scale", name) and len(parts) > 1:
        written |= registers_named(parts[1])
    return written


class Kernel:
    def __init__(self):
        self.code, self.before = [], []  # (mnemonic, operands); indexes of the instructions that may run just before

    def link(self, addresses, targets):
        place = {address: i for i, address in enumerate(addresses)}
        self.before = [[i - 1] if i and self.code[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64") else []
                       for i in range(len(self.code))]
        for i, target in targets:
            self.before[place[target]].append(i)

    def written_late(self, at, states, registers, writes):
        """Whether, on some way to `at`, the last write of one of the registers is one that `writes` finds, fewer than
        `states` wait states before."""
        seen, todo = set(), [(j, states, frozenset(registers)) for j in self.before[at]]
        while todo:
            j, left, open_ones = todo.pop()
            if left <= 0 or not open_ones or (j, left, open_ones) in seen:
                continue
            seen.add((j, left, open_ones))
            name, operands = self.code[j]
            if writes(name, operands) & open_ones:
                return True
            if name.startswith("s_") and not name.startswith(("s_cmp", "s_bitcmp", "s_cbranch")):
                open_ones -= registers_named(operands.split(", ")[0])
            passed = int(operands, 0) + 1 if name == "s_nop" else 1
            todo += [(k, left - passed, open_ones) for k in self.before[j]]
        return False


def kernels(listing):
    kernel, addresses, targets, start, name = None, [], [], 0, ""
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:$", line)
        if head:
            if kernel and kernel.code:
                kernel.link(addresses, targets)
                yield name, kernel
            kernel, addresses, targets, start, name = Kernel(), [], [], int(head[1], 16), head[2]
            continue
        found = LINE.match(line)
        if not found or kernel is None:
            continue
        if found[1].startswith(("s_cbranch", "s_branch")):
            targets.append((len(kernel.code), start + int(found[5] or "0", 16)))
        kernel.code.append((found[1], found[2]))
        addresses.append(int(found[3], 16))
    if kernel and kernel.code:
        kernel.link(addresses, targets)
        yield name, kernel


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    if not LIBRARY.exists():
        build.build()
    folder = tmp_path_factory.mktemp("listing")
    copy = shutil.copy(LIBRARY, folder / "library.so")  # the code objects are extracted beside it
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, capture_output=True, cwd=folder)
    found = {}
    for code in sorted(folder.glob("*gfx950*")):
        listing = subprocess.run([OBJDUMP, "-d", str(code)], check=True, capture_output=True, text=True).stdout
        if "global_load_lds" in listing:
            found.update(kernels(listing))
    return found


def copies(built):
    for name, kernel in built.items():
        for i, (mnemonic, operands) in enumerate(kernel.code):
            if mnemonic.startswith("global_load_lds"):
                yield name, kernel, i, operands


def scalar_m0(name, operands):
    return {"m0"} if name.startswith("s_") and operands.startswith("m0,") else set()


def test_a_wait_state_between_m0_and_the_copy(built):
    late = [f"{name} #{i}" for name, kernel, i, _ in copies(built) if kernel.written_late(i, 1, {"m0"}, scalar_m0)]
    assert sum(1 for _ in copies(built)) > 100
    assert not late, f"{len(late)} copies: {late[:5]}"


def test_five_wait_states_between_a_vector_write_and_the_copys_address(built):
    late = [f"{name} #{i}" for name, kernel, i, operands in copies(built)
            if kernel.written_late(i, 5, registers_named(operands), written_by_vector)]
    assert not late, f"{len(late)} copies: {late[:5]}"


def test_the_reading_itself():
    listing = """
0000000000001000 <k>:
\tv_readfirstlane_b32 s4, v1                                 // 000000001000: 00000000
\tv_readfirstlane_b32 s6, v1                                 // 000000001004: 00000000
\ts_mov_b32 m0, s9                                           // 000000001008: 00000000
\ts_add_u32 s6, s7, s8                                       // 00000000100C: 00000000
\ts_cbranch_scc1 2                                           // 000000001010: 00000000 <k+0x1c>
\ts_nop 2                                                    // 000000001014: 00000000
\ts_nop 0                                                    // 000000001018: 00000000
\tglobal_load_lds_dwordx4 v0, s[4:5]                         // 00000000101C: 00000000
\ts_endpgm                                                   // 000000001020: 00000000
"""
    (_, kernel), = kernels(listing)
    assert sorted(kernel.before[7]) == [4, 6]
    assert kernel.written_late(7, 5, {4, 5}, written_by_vector) and not kernel.written_late(7, 4, {4, 5}, written_by_vector)
    assert not kernel.written_late(7, 9, {6, 7}, written_by_vector)  # a scalar instruction wrote it since
    assert kernel.written_late(7, 3, {"m0"}, scalar_m0) and not kernel.written_late(7, 2, {"m0"}, scalar_m0)
