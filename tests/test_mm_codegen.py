"""mm_bf16's products are asm (kandinsky.cpp_amd/csrc/kd_mm_kernel.hip), so
that the compiler does not know the wait states around them: in the compiled
kernel, on every path, nothing but products touches an accumulator between
the first product and the wait behind the last, which the accumulators pass
one by one, and no vector instruction writes an operand within two wait
states ahead of the product that reads it."""
import re

import pytest

from kernel_asm import kernels, successors

TILES = {4: 64, 2: 32}   # accumulator blocks of a wave


def _instances():
    return [n for n in kernels("kd_mm_kernel.hip") if "mm_bf16" in n]


def _regs(text):
    out = set()
    for kind, lo, hi in re.findall(r"\b([av])\[(\d+):(\d+)\]", text):
        out |= {kind + str(r) for r in range(int(lo), int(hi) + 1)}
    return out | {k + r for k, r in re.findall(r"\b([av])(\d+)\b", text)}


def test_every_instance_is_checked():
    assert len(_instances()) == 4   # F32 and BF16 x, 256 and 128 tokens


@pytest.mark.parametrize("which", range(4))
def test_accumulators_wait_for_the_products(which):
    name = _instances()[which]
    lines = kernels("kd_mm_kernel.hip")[name]
    nxt = successors(lines)
    mfma = [i for i, ln in enumerate(lines) if ln.startswith("v_mfma")]
    acc = set().union(*(_regs(lines[i].split(", ")[0]) for i in mfma))
    blocks = TILES[4 if "Li4E" in name else 2]
    assert len(acc) == 4 * blocks and all(r[0] == "a" for r in acc)
    marks = [i for i, ln in enumerate(lines) if ln == "; accumulator complete"]
    assert len(marks) == blocks
    # from the products on, up to the markers: no other use of an accumulator,
    # and the markers are reached by way of the wait only
    todo, seen, met = [(j, False) for i in mfma for j in nxt[i]], set(), set()
    while todo:
        i, waited = todo.pop()
        if (i, waited) in seen:
            continue
        seen.add((i, waited))
        ln = lines[i]
        if ln == "; accumulator complete":
            assert waited
            met.add(i)
            if i == marks[-1]:
                continue
        elif ln == "s_nop 15":
            waited = True
        elif ln.startswith("v_mfma"):
            waited = False
        else:
            assert ln.startswith(";") or not _regs(ln) & acc, f"line {i}: {ln}"
        todo += [(j, waited) for j in nxt[i]]
    assert met == set(marks)


@pytest.mark.parametrize("which", range(4))
def test_operands_are_not_written_just_ahead_of_a_product(which):
    lines = kernels("kd_mm_kernel.hip")[_instances()[which]]
    before = {}
    for i, js in enumerate(successors(lines)):
        for j in js:
            before.setdefault(j, []).append(i)
    for i, ln in enumerate(lines):
        if not ln.startswith("v_mfma"):
            continue
        operands, todo = _regs(ln), [(p, 0) for p in before[i]]
        while todo:
            j, states = todo.pop()
            up = lines[j]
            if up.startswith("v_") and not up.startswith(("v_mfma", "v_cmp")):
                assert not _regs(up.split(", ")[0]) & operands, f"line {j}: {up} ahead of {ln}"
            if re.match(r"s_nop (\d+)", up):
                states += int(up.split()[1])
            states += not up.startswith((";", "."))
            if states < 2:
                todo += [(p, states) for p in before.get(j, [])]


@pytest.mark.parametrize("which", range(4))
def test_every_step_loads_its_share_of_f32_x(which):
    """The waits count on the loads and DMAs of each step, F32 x's plain loads
    among them: none merged, dropped or added (two stages ahead of the loop
    and two behind its first rounding, then one per step of the two loops;
    the single last step has none)."""
    name = _instances()[which]
    lines = kernels("kd_mm_kernel.hip")[name]
    end = lines.index("; accumulator complete")
    loads = sum(ln.startswith("global_load_dwordx4") for ln in lines[:end])
    dmas = sum(ln.startswith("global_load_lds_dwordx4") for ln in lines[:end])
    mb = 4 if "Li4E" in name else 2
    if "Lb1E" in name:
        assert (loads, dmas) == (2 * mb * (4 + 4), 3 * 8 + 5 * 4)
    else:
        ahead = (5 if mb == 4 else 6) - 1
        per = 4 + mb
        assert (loads, dmas) == (0, ahead * per + (2 + mb // 2) + 5 * per)
