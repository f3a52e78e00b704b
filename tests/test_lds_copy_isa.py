"""Copies memory-to-LDS in the generated code of the built library. They are inline assembly, which
the compiler's hazard handling does not look into, so what precedes each is checked here:

- m0 (the LDS address) is written at least one wait state before a copy;
- a scalar base is not written by a vector instruction (a readlane, say) within five wait states;
- the images of the f16 prefill mode, whole groups of four KiB per wave, take one write of m0 (and
  one wait) per four copies.
"""
import os
import re
import subprocess

import pytest

import eyebrowse_amd as eb

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def _sgprs(text):
    """The scalar registers that an operand list names."""
    out = set()
    for a, lo, hi in re.findall(r"\bs(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        out |= {int(a)} if a else set(range(int(lo), int(hi) + 1))
    return out


def _check(ins, i):
    """What is wrong with the copy ins[i] (None: nothing). ins: (mnemonic, operands) in order; a
    branch in between is read straight through."""
    base = _sgprs(ins[i][1])
    states = 0  # wait states between the instruction looked at and the copy
    for op, args in reversed(ins[max(0, i - 8):i]):
        dst = args.split(",")[0]
        if dst == "m0" and states < 1:
            return "m0 written right before it"
        if op.startswith("v_") and states < 5 and base & _sgprs(dst):
            return f"scalar base written by {op} {states} wait states before it"
        states += 1 + (int(args) if op == "s_nop" else 0)
    return None


def test_the_check_sees_both_hazards():
    copy = ("global_load_lds_dwordx4", "v2, s[4:5]")
    m0, nop = ("s_mov_b32", "m0, s8"), ("s_nop", "0")
    lane = ("v_readfirstlane_b32", "s5, v1")
    assert _check([m0, nop, copy], 2) is None
    assert _check([m0, copy], 1)
    assert _check([lane, m0, nop, copy], 3)
    assert _check([lane, m0, ("s_nop", "3"), copy], 3) is None
    assert _check([("v_readfirstlane_b32", "s6, v1"), m0, nop, copy], 3) is None


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> [(mnemonic, operands)] of every kernel with such copies."""
    d = tmp_path_factory.mktemp("isa")
    eb.lib()  # (says how to build it if it is missing)
    src = os.path.join(os.path.dirname(os.path.abspath(eb.__file__)), "libeyebrowse_hip.so")
    os.symlink(src, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    out, name = {}, None
    for f in sorted(d.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True,
                              capture_output=True, text=True).stdout
        if "_load_lds" not in text:
            continue
        for line in text.splitlines():
            if line.endswith(">:"):
                name = line.split("<")[1][:-2]
                out[name] = []
            elif line.startswith("\t") and name:
                op, _, args = line.split("//")[0].strip().partition(" ")
                out[name].append((op, args.strip()))
    return {n: ins for n, ins in out.items() if any("_load_lds" in op for op, _ in ins)}


def test_no_hazard_before_a_copy(kernels):
    assert any("linear_tile_kernel" in n for n in kernels)
    assert any("prefill_kernel" in n for n in kernels)
    for n, ins in kernels.items():
        for i, (op, _) in enumerate(ins):
            if "_load_lds" in op:
                assert _check(ins, i) is None, (n, _check(ins, i))


def test_one_m0_write_per_four_copies(kernels):
    # prefill_kernel<128, 4 waves, no key split, records, f16 mode>: 16 KiB images
    fast = [n for n in kernels if re.search(r"prefill_kernelILi128ELi[124]ELi[124]ELi1ELb0ELi4ELb1ELb1E", n)]
    assert fast
    for n in fast:
        copies = sum("_load_lds" in op for op, _ in kernels[n])
        writes = sum(args.startswith("m0,") for _, args in kernels[n])
        assert copies == 4 * writes, (n, copies, writes)
