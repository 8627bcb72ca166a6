"""Wait states that hand-written instructions keep by themselves: the compiler places none for what it cannot see."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parent.parent / "dynaflow_amd" / "csrc"


def wait_states(instructions):
    return sum(int(i.split()[1]) + 1 if i.startswith("s_nop") else 1 for i in instructions)


def test_the_exchange_of_neighbours_waits_on_both_sides():
    """Two states between a vector write and a read of the register by another lane, and between one and an MFMA that reads it,
    whatever the compiler puts next to the block."""
    source = (CSRC / "dfhip_common.h").read_text()
    body = source[source.index("void deal_neighbours("):]
    block = body[body.index("asm("):body.index(': "=&v"')]
    block = re.sub(r"//[^\n]*", "", block)
    text = "".join(re.findall(r'"([^"]*)"', block))
    instructions = [i.strip() for i in text.replace("\\t", "").split("\\n")]
    vector = [i for i, line in enumerate(instructions) if line.startswith("v_")]
    assert len(vector) == 8
    assert wait_states(instructions[:vector[0]]) >= 2
    assert wait_states(instructions[vector[-1] + 1:]) >= 2
