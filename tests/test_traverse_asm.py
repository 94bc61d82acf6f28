"""The traversals' assembly blocks, read as text: the first v_readlane, whose lane number comes from a vector
instruction before the block, has the four wait states that this needs."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "batchlayoutcode_amd", "csrc")


def _read(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


def _instructions(text):
    """The instructions of the string literals that are assembly, in order."""
    out = []
    for lit in re.findall(r'"((?:[^"\\]|\\.)*)"', text):
        out += [i.strip() for i in re.split(r"\\n\\t|\\n|\\t", lit) if re.match(r"\s*[sv]_[a-z0-9_]+", i)]
    return out


def test_wait_states_before_the_first_readlane():
    text = _read("traverse.h")
    pop = text[text.index("#define BL_TRAV_POP"):text.index("// (dx, dy) = c - p")]
    states = 0
    for ins in _instructions(pop):
        if ins.startswith("v_readlane"):
            break
        nop = re.fullmatch(r"s_nop (\d+)", ins)
        states += int(nop.group(1)) + 1 if nop else 1
    else:
        raise AssertionError("no v_readlane")
    assert states >= 4
