"""Waits in the code of kernels whose matrix products are inline assembly: the compiler puts none between such a product and its neighbours."""
import os
import re
import struct
import subprocess

import pytest

from scaling_amd.csrc.build import LIB_PATH

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
OPERAND = 2                                                # wait states between a vector instruction's result and a product that takes it


def _code_objects(path):
    data = open(path, "rb").read()
    for found in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        start = found.start()
        at = start + 32
        for _ in range(struct.unpack_from("<Q", data, start + 24)[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, at)
            if size and b"gfx950" in data[at + 24:at + 24 + name]:
                yield data[start + offset:start + offset + size]
            at += 24 + name


def _registers(operand):
    """v and a registers of an operand, as a set of (kind, number)"""
    found = re.fullmatch(r"[-|]*([va])(?:(\d+)|\[(\d+):(\d+)\])\|?", operand.strip())
    if not found:
        return frozenset()
    first, last = (int(found[2]),) * 2 if found[2] else (int(found[3]), int(found[4]))
    return frozenset((found[1], n) for n in range(first, last + 1))


class _Instruction:
    def __init__(self, line):
        text, _, rest = line.partition("//")
        self.text = text.strip()
        self.name, _, operands = self.text.partition(" ")
        self.operands = [_registers(o.split()[0] if o.split() else "") for o in operands.split(",")]
        self.uses = frozenset().union(*self.operands)
        self.matrix = "_mfma_" in self.name
        self.vector = self.name.startswith("v_") and not self.matrix
        self.address = int(rest.split(":")[0], 16)
        target = re.search(r"<\S+\+0x([0-9a-f]+)>", rest)
        self.target = int(target[1], 16) if target and "branch" in self.name else None
        self.states = int(operands, 0) + 1 if self.name == "s_nop" else 1


def _function(lines):
    code = [_Instruction(line) for line in lines if "//" in line]
    at = {i.address - code[0].address: n for n, i in enumerate(code)}
    after = [[n + 1] if i.name not in ("s_branch", "s_endpgm") and n + 1 < len(code) else [] for n, i in enumerate(code)]
    for n, i in enumerate(code):
        if i.target is not None:
            after[n].append(at[i.target])
    return code, after


def _early(code, after, n, limit, passes, meets):
    """Instructions that `meets` names and that some way through the code reaches less than `limit` wait states behind instruction n; a product starts `passes`
    behind another at the soonest"""
    found, best = [], {}
    todo = [(m, 0, 0 if code[n].matrix else -passes) for m in after[n]]     # where, states since n, when the last product started
    while todo:
        m, states, product = todo.pop()
        i = code[m]
        if i.matrix:
            states = max(states, product + passes)
        if states >= limit or best.get(m, (limit, 0)) <= (states, -product):
            continue
        best[m] = (states, -product)
        if meets(i):
            found.append((states, i.text))
        todo += [(k, states + i.states, states if i.matrix else product) for k in after[m]]
    return found


def _kernels(pattern):
    for code in _code_objects(LIB_PATH):
        if pattern.encode() not in code:
            continue
        listing = subprocess.run([OBJDUMP, "-d", "-"], input=code, capture_output=True, check=True).stdout.decode()
        for name, body in re.findall(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^\n|\Z)", listing, re.M | re.S):
            if pattern in name:
                yield name, _function(body.splitlines())


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(LIB_PATH)), reason="no library, or nothing to list its code with")
# kernels, their products, the passes that one takes at least, wait states between it and another instruction's use of its result
@pytest.mark.parametrize("pattern,count,product,passes,states", [
    ("attn_f32_dkdv_kernel", 11, r"v_mfma_f32_32x32x2_f32", 16, 18), ("11wide_kernelI", 4, r"v_mfma_f32_16x16x32_b?f16", 4, 12),
])
def test_products_and_their_neighbours(pattern, count, product, passes, states):
    """Nothing reads or overwrites a product's result, and no product takes a vector instruction's, too early."""
    kernels = dict(_kernels(pattern))
    assert len(kernels) >= count
    for name, (code, after) in kernels.items():
        assert any(i.matrix for i in code), name
        for n, i in enumerate(code):
            result = i.operands[0]
            if i.matrix:
                assert re.fullmatch(product, i.name), i.text
                # a product that adds to the whole of it may follow at once
                early = _early(code, after, n, states, passes, lambda j: (result & j.uses) and not (
                    j.matrix and j.operands[0] == result and j.operands[3] in (result, frozenset()) and not result & (j.operands[1] | j.operands[2])))
            elif i.vector and result:
                early = _early(code, after, n, OPERAND, passes, lambda j: j.matrix and result & (j.operands[1] | j.operands[2] | j.operands[3]))
            else:
                continue
            assert not early, f"{name}: {i.text}: {early}"
