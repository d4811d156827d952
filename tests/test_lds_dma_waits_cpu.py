"""No barrier is passed with an LDS DMA in flight, shown on the built code objects: a fixed point over each kernel's control
flow.  Only `s_waitcnt vmcnt(0)` lands a DMA: a counted wait that covered the older DMA and left younger loads in flight has
let readers see rows that had not arrived.  The compiler counts wherever it can tell the loads apart, so the full wait has to
be in the source (w4_dma_barrier).  The decode kernel's DMA is wave-private and passes no barrier; it is not looked at here."""
import os
import re
import subprocess

import pytest

from llm170_amd import build

OBJDUMP = os.path.join(build.ROCM, "llvm", "bin", "llvm-objdump")
KERNEL = re.compile(r"^([0-9a-f]+) <([^>]+)>:$")
INSN = re.compile(r"^\s+(\S+)(.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<([^+>]+)(?:\+0x([0-9a-f]+))?>)?$")


def kernels(text):
    """name -> list of (address, mnemonic, operands, branch target or None), in address order."""
    out, at = {}, {}
    for line in text.splitlines():
        m = KERNEL.match(line)
        if m:
            cur = out.setdefault(m.group(2), [])
            at[m.group(2)] = int(m.group(1), 16)
            continue
        m = INSN.match(line)
        if m:
            target = at[m.group(4)] + int(m.group(5) or "0", 16) if m.group(4) else None
            cur.append((int(m.group(3), 16), m.group(1), m.group(2), target))
    return out


def open_barriers(insns):
    """Addresses of the barriers that some path reaches with an LDS DMA in flight, and the number of DMA instructions."""
    index = {a: i for i, (a, _, _, _) in enumerate(insns)}
    dma = [mn.startswith("buffer_load") and ops.split()[-1:] == ["lds"] for _, mn, ops, _ in insns]
    seen, bad, work = set(), set(), [(0, False)]
    while work:
        i, pending = work.pop()
        while (i, pending) not in seen:
            seen.add((i, pending))
            addr, mn, ops, target = insns[i]
            if dma[i]:
                pending = True
            elif mn == "s_waitcnt" and "vmcnt(0)" in ops:
                pending = False
            elif mn == "s_barrier" and pending:
                bad.add(addr)
            assert not mn.startswith(("s_setpc", "s_swappc", "s_call")), "a call the walk does not follow"
            if mn == "s_endpgm":
                break
            if mn.startswith(("s_branch", "s_cbranch")):
                work.append((index[target], pending))
                if mn == "s_branch":
                    break
            i += 1
    return bad, sum(dma)


def test_walk_tells_the_waits_apart():
    line = "\t%s // %012X: 00000000%s"
    def text(wait):
        body = ["buffer_load_dwordx4 v1, s[0:3], 0 offen lds", "buffer_load_dwordx4 v[4:7], v1, s[0:3], 0 offen", wait, "s_barrier",
                "s_cbranch_scc1 65531", "s_endpgm"]
        return "\n".join(["0000000000000100 <k>:"] + [line % (b, 0x100 + 4 * i, " <k+0x0>" if "branch" in b else "") for i, b in enumerate(body)])
    assert open_barriers(kernels(text("s_waitcnt vmcnt(0) lgkmcnt(0)"))["k"]) == (set(), 1)
    assert open_barriers(kernels(text("s_waitcnt vmcnt(1)"))["k"]) == ({0x10C}, 1)


@pytest.mark.parametrize("asset,least", [("mid", 96), ("moe", 32), ("prefill", 20), ("prefill_g128", 20)])
def test_no_barrier_with_lds_dma_in_flight(asset, least):
    """`least`: kernels of the code object that use LDS DMA (mid.hip: eight of eleven builds of each family at least)."""
    text = subprocess.run([OBJDUMP, "-d", os.path.join(build.ASSET_DIR, asset + ".hsaco")], stdout=subprocess.PIPE, text=True, check=True).stdout
    users, bad = 0, {}
    for name, insns in kernels(text).items():
        found, dma = open_barriers(insns)
        users += dma > 0
        if found:
            bad[name] = sorted(hex(a) for a in found)
    assert users >= least, users
    assert not bad, (len(bad), sorted(bad.items())[:4])
