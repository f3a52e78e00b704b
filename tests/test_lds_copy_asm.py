"""Copies memory-to-LDS written as inline assembly: m0 (their LDS address) is written one wait
state before the copy at the soonest. The compiler inserts none inside an asm block."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parent.parent / "eyebrowse_amd" / "csrc"


def test_a_wait_state_between_m0_and_the_copy():
    copies = 0
    for f in sorted(CSRC.glob("*.hip")):
        for asm in re.findall(r'asm volatile\("([^"]*)"', f.read_text()):
            ins = asm.split("\\n\\t")
            for before, here in zip([""] + ins, ins):
                if here.startswith(("global_load_lds", "buffer_load_lds")):
                    copies += 1
                    assert before.startswith("s_nop"), f"{f.name}: {asm}"
    assert copies
