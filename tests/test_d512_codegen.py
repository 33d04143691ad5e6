"""fa_fwd_d512's one K buffer (kandinsky.cpp_amd/csrc/kd_fa_d512.hip) is
refilled by DMAs written in asm: in the compiled kernel, on every path, the
reads of K's fragments have returned, and the source says so to the compiler
(its marker), before the first DMA that follows them."""
import re

import pytest

from kernel_asm import kernels, successors


def _names():
    return [n for n in kernels("kd_fa_d512.hip") if "fa_fwd_d512" in n]


def test_every_instance_is_checked():
    assert len(_names()) == 4   # BF16 and F16, 32 and 64 rows


@pytest.mark.parametrize("which", range(4))
def test_k_reads_return_before_the_refill(which):
    lines = kernels("kd_fa_d512.hip")[_names()[which]]
    nxt = successors(lines)
    # K's fragments: the eight 16-byte reads that follow the wait for K's DMAs
    # (all of them in the prologue, all but V's eight in the loop)
    k_reads = set()
    for i, ln in enumerate(lines):
        if ln in ("s_waitcnt vmcnt(0)", "s_waitcnt vmcnt(8)") and lines[i - 1] == ";;#ASMSTART":
            after = [j for j in range(i + 1, len(lines)) if lines[j].startswith("ds_read_b128")][:8]
            upto = after[-1] if len(after) == 8 else len(lines)
            if not any(re.match(r"ds_read_b64|ds_read_b32|s_barrier|buffer_load", ln) for ln in lines[i + 1:upto]):
                k_reads.update(after)
    assert len(k_reads) == 8 * 3, len(k_reads)   # prologue, the loop's first tile (peeled), the loop
    # K's DMAs: those with the offset registers of the first tile's eight (the
    # kernel's first DMAs; V's, the next eight and issued before the first
    # wait, share no register with them)
    dma = [(i, ln.split()[1]) for i, ln in enumerate(lines) if ln.startswith("buffer_load") and ln.endswith(" lds")]
    k_off = {r for _, r in dma[:8]}
    k_dma = {i for i, r in dma if r in k_off}
    assert len(k_off) == 8 and not k_off & {r for _, r in dma[8:16]}
    assert dma[15][0] < min(k_reads)
    assert len(k_dma) == 8 * 5   # the prologue's two tiles, the first tile (peeled), the loop's two branches
    reached = set()
    # state: line, K reads since a marker, LDS operations in flight (True: a read of K), oldest first
    todo, seen = [(0, False, ())], set()
    while todo:
        state = todo.pop()
        if state in seen:
            continue
        seen.add(state)
        assert len(seen) < 2_000_000
        i, read, flight = state
        ln = lines[i]
        if i in k_reads:
            read, flight = True, flight + (True,)
        elif ln.startswith("ds_"):
            flight = flight + (False,)
        elif ln.startswith("s_waitcnt"):
            m = re.search(r"lgkmcnt\((\d+)\)", ln)
            if m:
                flight = flight[max(0, len(flight) - int(m.group(1))):]
        elif ln == "; K fragments held":
            assert not any(flight), f"line {i}: a read of K may be in flight"
            read = False
        elif i in k_dma:
            assert not read, f"line {i}: {ln} after a read of K, and no marker between"
            reached.add(i)
        if True not in flight:
            flight = ()
        todo += [(j, read, flight) for j in nxt[i]]
    assert reached == k_dma


@pytest.mark.parametrize("which", range(4))
def test_one_tile_fetches_one_tile(which):
    """A range of one key tile (a split short call is all such) brings that
    tile's K and V and nothing else: the fewest DMAs of any path on from the
    first."""
    lines = kernels("kd_fa_d512.hip")[_names()[which]]
    nxt = successors(lines)
    dma = [ln.startswith("buffer_load") and ln.endswith(" lds") for ln in lines]
    first = dma.index(True)
    least, todo = {first: 1}, [first]
    while todo:
        i = todo.pop()
        for j in nxt[i]:
            if least[i] + dma[j] < least.get(j, len(lines)):
                least[j] = least[i] + dma[j]
                todo.append(j)
    assert min(n for i, n in least.items() if lines[i].startswith("s_endpgm")) == 16
