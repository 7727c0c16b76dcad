"""The inline assembly's operands.  Carries: an instruction that reads a carry
has at least two others, or as many wait states, after the vector instruction
that wrote it (the distance the compiler keeps on gfx950 between its own),
within the same block.  Registers: an operand that a block writes before it
has read all the others is early clobber, so that no other shares its place."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "zkmetal_amd", "csrc")
READS = ("v_addc_co_u32", "v_subb_co_u32", "v_subbrev_co_u32", "v_cndmask_b32")
WRITES = ("v_mad_u64_u32", "v_add_co_u32", "v_sub_co_u32", "v_subrev_co_u32") + READS[:3]


def blocks(text):
    """instruction lists of the asm statements, macros of strings expanded"""
    text = text.replace("\\\n", " ")
    macros = {}
    for name, args, body in re.findall(r"^#define (\w+)\(([^)]*)\)((?: *(?:\"[^\"]*\"|#\w+))+) *$", text, re.M):
        macros[name] = ([a.strip() for a in args.split(",")], body)

    def expand(m):
        args, body = macros[m.group(1)]
        for a, v in zip(args, m.group(2).split(",")):
            body = re.sub(r"#%s\b" % a, '"%s"' % v.strip(), body)
        return body

    for m in re.finditer(r"\basm(?: volatile)?\(", text):
        part = text[m.end():]
        for name in macros:
            part = re.sub(r"\b(%s)\(([^)]*)\)" % name, expand, part[:4000])
        head = re.match(r"(?:\s*\"(?:[^\"\\]|\\.)*\")*", part).group(0)
        code = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", head))
        outs = re.findall(r"(?:\"([^\"]*)\"|\bY)\s*\(", part[len(head):].split(";")[0])
        yield [i.strip() for i in re.split(r"\\n|\\t", code) if i.strip()], outs


def short_waits(block):
    age, out = {}, []
    for ins in block:
        op, _, rest = ins.partition(" ")
        a = [x.strip() for x in rest.split(",")]
        op = re.sub(r"_e(32|64)$", "", op)
        if op == "s_nop":
            age = {r: n + int(a[0]) + 1 for r, n in age.items()}
            continue
        if op in READS and age.get(a[-1], 0) < 2:  # (no writer in the block: too near as well)
            out.append(ins)
        age = {r: n + 1 for r, n in age.items()}
        if op in WRITES:
            age[a[1]] = 0
    return out


@pytest.mark.parametrize("name", sorted(os.path.basename(p) for p in glob.glob(os.path.join(CSRC, "*.h*"))))
def test_carries_are_read_in_time(name):
    for block, _ in blocks(open(os.path.join(CSRC, name)).read()):
        assert not short_waits(block), block


def shared(block, constraints):
    """operands written while others are still to be read, not early clobber"""
    out = []
    for k, ins in enumerate(block):
        for d in re.findall(r"^v_\S+ %(\d+),", ins):
            later = {int(x) for i in block[k + 1:] for x in re.findall(r"%(\d+)", i.partition(",")[2])}
            inputs = {x for x in later if x < len(constraints) and not constraints[x].startswith(("+", "="))}
            if inputs and "&" not in constraints[int(d)]:
                out.append(ins)
    return out


@pytest.mark.parametrize("name", sorted(os.path.basename(p) for p in glob.glob(os.path.join(CSRC, "*.h*"))))
def test_written_operands_share_no_register(name):
    for block, constraints in blocks(open(os.path.join(CSRC, name)).read()):
        assert not shared(block, constraints), (block, constraints)


def test_the_check_sees_the_products():
    found = [b for b, _ in blocks(open(os.path.join(CSRC, "field.hpp")).read()) if any("addc" in i for i in b)]
    assert sorted(sum("v_mad_u64_u32" in i for i in b) for b in found) == [1, 2, 3]
    assert short_waits(["v_mad_u64_u32 %0, vcc, %2, %3, %0", "v_addc_co_u32 %1, vcc, 0, %1, vcc"])
    assert short_waits(["v_mad_u64_u32 %0, %2, %3, %4, %0", "s_nop 0", "v_addc_co_u32_e64 %1, %2, 0, %1, %2"])
