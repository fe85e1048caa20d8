"""The tiled contraction issues its 16x16x64 products from inline assembly, where the compiler does not see to the wait states around them.
Which registers they take, and what is scheduled between them, is the compiler's choice: this reads the assembly that it writes for this
source and follows every path around every product."""
import os
import re
import shutil
import subprocess

import pytest

from matmulfreellm_amd import build

READ = 16          # wait states until a product's result may be read or replaced by anything but the next product (8 passes: 11)
WRITE = 2          # wait states from a vector operation's result to a product that reads it
PRODUCT = "v_mfma_i32_16x16x64_i8"


def _registers(operand):
    regs = set()
    for first, last, one in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", operand):
        regs |= set(range(int(first), int(last) + 1)) if first else {int(one)}
    return regs


class Instruction:
    def __init__(self, text):
        self.op, _, rest = text.partition(" ")
        self.operands = [o.strip() for o in rest.split(",")] if rest.strip() else []
        self.waits = int(self.operands[0], 0) + 1 if self.op == "s_nop" else 1
        self.product = self.op == PRODUCT
        self.registers = [_registers(o) for o in self.operands]
        self.target = self.operands[0] if self.op.startswith(("s_cbranch", "s_branch")) else None

    @property
    def all(self):
        return set().union(*self.registers) if self.registers else set()

    @property
    def writes(self):
        """Vector operations write their first operand, the exchange of half-waves both."""
        if not self.op.startswith("v_") or self.op.startswith(("v_cmp", "v_readfirstlane", "v_readlane")) or not self.registers:
            return set()
        return self.registers[0] | (self.registers[1] if self.op.startswith(("v_swap", "v_permlane")) else set())


def _kernels(text):
    """name -> (instructions, index of every label)."""
    name, out = None, {}
    for line in text.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"^([\w.$]+):", line)
        if label and not label[1].startswith(".L"):
            name = label[1] if "bitlinear_mfma_dma3_kernel" in label[1] else None
            if name:
                out[name] = ([], {})
        elif label and name:
            out[name][1][label[1]] = len(out[name][0])
        elif name and line and not line.startswith((".", "//")):
            out[name][0].append(Instruction(line))
        if line.startswith(".section") or line.startswith(".end_amdhsa_kernel"):
            name = None
    return out


def _next(code, labels, i):
    """The instructions that can follow number i."""
    if code[i].op in ("s_endpgm", "s_setpc_b64"):
        return []
    to = [labels[code[i].target]] if code[i].target else []
    return to if code[i].op == "s_branch" else to + [i + 1]


def _faults(code, labels):
    found = []
    before = {i: [] for i in range(len(code) + 1)}
    for i in range(len(code)):
        for j in _next(code, labels, i):
            if j < len(code):
                before[j].append(i)
    for i, ins in enumerate(code):
        if ins.op.startswith("scratch_"):
            found.append((i, "a register spilled"))
        if not ins.product:
            continue
        result = ins.registers[0]
        if result != ins.registers[3]:
            found.append((i, "accumulates elsewhere"))
        todo, seen = [(j, READ) for j in _next(code, labels, i)], {}
        while todo:                                                    # forwards: nobody touches the result too early
            j, left = todo.pop()
            if left <= 0 or j >= len(code) or seen.get(j, 0) >= left:
                continue
            seen[j] = left
            other = code[j]
            if other.product:
                if other.registers[0] != result and other.all & result or (other.registers[1] | other.registers[2]) & result:
                    found.append((j, "a product reads another's result too early"))
            elif other.all & result:
                found.append((j, f"{other.op} touches a result too early"))
            todo += [(k, left - other.waits) for k in _next(code, labels, j)]
        todo, seen = [(j, WRITE) for j in before[i]], {}
        while todo:                                                    # backwards: nobody has just written what it reads
            j, left = todo.pop()
            if left <= 0 or seen.get(j, 0) >= left:
                continue
            seen[j] = left
            if not code[j].product and code[j].writes & ins.all:
                found.append((j, f"{code[j].op} writes an operand too late"))
            todo += [(k, left - code[j].waits) for k in before[j]]
    return found


def test_the_reader_finds_a_planted_hazard():
    good = "k_bitlinear_mfma_dma3_kernel:\n v_and_b32_e32 v4, 3, v9\n s_nop 1\n" + f" {PRODUCT} v[0:3], v[4:7], v[8:11], v[0:3]\n s_nop 15\n s_nop 15\n v_mov_b32_e32 v20, v0\n s_endpgm\n"
    assert [len(c) for c, _ in _kernels(good).values()] == [7]
    assert not any(_faults(*k) for k in _kernels(good).values())
    for bad in (good.replace(" s_nop 1\n", " s_nop 0\n"), good.replace(" s_nop 15\n s_nop 15\n", " s_nop 9\n"),
                good.replace(" s_nop 15\n", " v_mov_b32_e32 v3, 0\n", 1), good.replace("v[0:3]\n", "v[12:15]\n"),
                good.replace(" s_nop 15\n", " scratch_store_dword off, v30, off\n", 1)):
        assert all(_faults(*k) for k in _kernels(bad).values()), bad


@pytest.mark.skipif(not shutil.which(build._hipcc()), reason="no hipcc here: the library was built elsewhere")
def test_products_of_the_tiled_contraction_have_their_wait_states(tmp_path):
    out = tmp_path / "bitlinear_mfma.s"
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, "bitlinear_mfma.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    kernels = _kernels(out.read_text())
    products = {name: sum(i.product for i in code) for name, (code, _) in kernels.items()}
    assert sum(n > 0 for n in products.values()) >= 20, products
    faults = {name: _faults(*k)[:5] for name, k in kernels.items() if products[name]}
    assert not any(faults.values()), {n: f for n, f in faults.items() if f}
