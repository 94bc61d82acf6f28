"""The traversals' assembly blocks, read as text: every fixed register that an instruction writes is in the
clobber list, and the first v_readlane, whose lane number comes from a vector instruction before the block,
has the four wait states that this needs."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "batchlayoutcode_amd", "csrc")
NO_DEST = ("s_cmp", "s_cbranch", "s_branch", "s_nop", "s_waitcnt")


def _read(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


def _instructions(text):
    """The instructions of the string literals that are assembly, in order."""
    out = []
    for lit in re.findall(r'"((?:[^"\\]|\\.)*)"', text):
        out += [i.strip() for i in re.split(r"\\n\\t|\\n|\\t", lit) if re.match(r"\s*[sv]_[a-z0-9_]+", i)]
    return out


def _clobbers():
    text = _read("traverse.h")
    return set(re.findall(r'"([a-z0-9]+)"', text[text.index("#define BL_TRAV_CLOBBERS"):]))


def _written(ins):
    m = re.match(r"([sv]_[a-z0-9_]+)\s+([^,\s]+)", ins)
    if not m or m.group(1).startswith(NO_DEST):
        return set()
    dest = m.group(2)
    r = re.fullmatch(r"s\[(\d+):(\d+)\]", dest)
    if r:
        return {f"s{k}" for k in range(int(r.group(1)), int(r.group(2)) + 1)}
    return {dest} if re.fullmatch(r"s\d+|vcc|m0", dest) else set()


def test_written_registers_are_clobbers():
    bh, far = _read("bh.hip"), _read("farfield.hip")
    blocks = [_read("traverse.h")]
    i = bh.index("BL_TRAV_POP")
    blocks.append(bh[i:bh.index("BL_TRAV_CLOBBERS", i)])
    blocks.append(far[far.index("#define BL_FARTRAV_NODE"):far.index("#define BL_FARTRAV_LOOP")])
    ins = [i for b in blocks for i in _instructions(b)]
    assert len(ins) > 80
    written = set().union(*map(_written, ins))
    assert {"m0", "vcc", "s80", "s92"} <= written
    assert written <= _clobbers(), sorted(written - _clobbers())


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
