"""The matrix-core products that the prefill kernels issue from inline asm
(accumulators in accumulator registers), read from the built library: the
compiler keeps no distance around them, so the source has to. A product's
operands are not written by a vector instruction less than two wait states
before it, and its outputs are not touched by one less than 20 wait states
after it (a 16-pass product's; these have 8)."""

import re
import shutil
import subprocess

import pytest

from instinct_amd import _lib

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin") or shutil.which("llvm-objdump")
READ, WRITE = 2, 20  # wait states


def registers(text):
    """The vector and accumulator registers an operand list names."""
    out = set()
    for kind, a, b, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))", text):
        out |= {kind + str(i) for i in range(int(a or one), int(b or one) + 1)}
    return out


def parse(lines):
    """A kernel's instructions: (mnemonic, first operand's registers, the
    others', wait states, addresses it may come from)."""
    ops, at = [], {}
    for line in lines:
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):.*?(?:<\S+?\+0x([0-9a-f]+)>)?$", line)
        if m:
            at[int(m[3], 16)] = len(ops)
            ops.append((m[1], m[2], int(m[4], 16) if m[4] else None))
    base = min(at)
    out = []
    for i, (name, text, _) in enumerate(ops):
        first, _, rest = text.partition(",")
        falls = i > 0 and ops[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64")
        out.append((name, registers(first), registers(rest),
                    int(text.split()[0], 0) + 1 if name == "s_nop" else 1, [i - 1] if falls else []))
    for i, (name, _, target) in enumerate(ops):
        if name.startswith(("s_cbranch", "s_branch")) and target is not None:
            out[at[base + target]][4].append(i)
    return out


def behind(ops, start, states):
    """The instructions less than ``states`` wait states before ``start``, on
    any way to it."""
    seen, todo = {}, [(p, 0) for p in ops[start][4]]
    while todo:
        i, waited = todo.pop()
        if waited >= states or seen.get(i, states) <= waited:
            continue
        seen[i] = waited
        todo += [(p, waited + ops[i][3]) for p in ops[i][4]]
    return seen


def faults(ops):
    inline = {i for i, op in enumerate(ops)
              if "mfma" in op[0] and any(r[0] == "a" for r in op[1])}
    found = []
    for i, (name, first, rest, _, _) in enumerate(ops):
        if i in inline:
            found += [(j, i) for j in behind(ops, i, READ)
                      if ops[j][0].startswith("v_") and "mfma" not in ops[j][0]
                      and ops[j][1] & (first | rest)]
        elif name.startswith("v_") and "mfma" not in name:
            touched = {r for r in first | rest if r[0] == "a"}
            if touched:
                found += [(j, i) for j in behind(ops, i, WRITE)
                          if j in inline and ops[j][1] & touched]
    return found, len(inline)


def listing(*texts):
    """Text of the disassembler's form, 8 bytes an instruction."""
    return parse([f"\t{t}  // {8 * i:012X}: 00" for i, t in enumerate(texts)])


PRODUCT = "v_mfma_f32_32x32x16_f16 a[0:15], v[0:3], v[4:7], a[0:15]"


@pytest.mark.parametrize("before,after,count", [
    (["v_mov_b32_e32 v5, v9"], [], 1),
    (["v_mov_b32_e32 v5, v9", "s_nop 0"], [], 1),
    (["v_mov_b32_e32 v5, v9", "s_nop 1"], [], 0),
    (["v_accvgpr_write_b32 a3, v9", "v_mov_b32_e32 v9, v8"], [], 1),
    (["v_mov_b32_e32 v8, v5", "v_mov_b32_e32 v9, v8"], [], 0),
    ([], ["v_accvgpr_read_b32 v9, a15"], 1),
    ([], ["s_nop 15", "s_nop 2", "v_accvgpr_read_b32 v9, a15"], 1),
    ([], ["s_nop 15", "s_nop 3", "v_accvgpr_read_b32 v9, a15"], 0),
    ([], ["v_accvgpr_read_b32 v9, a16"], 0),
])
def test_planted(before, after, count):
    assert len(faults(listing(*before, PRODUCT, *after))[0]) == count


def test_planted_over_a_branch():
    ops = listing("v_mov_b32_e32 v5, v9", "s_nop 3", PRODUCT)
    assert not faults(ops)[0]
    ops[2][4].append(0)  # the product is a branch's target as well
    assert len(faults(ops)[0]) == 1


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_built_kernels(tmp_path):
    library = tmp_path / "lib.so"
    library.symlink_to(_lib.LIBRARY_PATH)
    subprocess.run([OBJDUMP, "--offloading", library.name], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    kernels = 0
    for image in sorted(tmp_path.glob("*gfx950*")):
        if b"prefill_pipe_kernel" not in image.read_bytes():
            continue
        text = subprocess.run([OBJDUMP, "-d", image.name], cwd=tmp_path, check=True,
                              capture_output=True, text=True).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text,
                                     re.S | re.M):
            if "prefill_pipe_kernel" not in name:
                continue
            found, products = faults(parse(body.splitlines()))
            assert not found, f"{name}: {found[:4]}"
            kernels += products > 0
    assert kernels == 4  # D = 256, and D = 128 with two query blocks; fp16 and bf16
