"""LDS reads written in inline asm (gemm.hip, gemm_tile.h, prefill.hip) are waited for apart from the
read, by count.  The compiler takes such a register as written at once, so nothing but the code's own
shape keeps it from copying, spilling or reusing one whose read is in flight.  Here the assembly of
this library's own build is walked along every branch: between a read and the wait that covers it no
instruction may name a register of it."""
import concurrent.futures as cf
import os
import re
import subprocess
import sys

import pytest

import __graft_entry__

sys.path.insert(0, __graft_entry__.PKG_DIR)
import build as hipbuild  # noqa: E402

sys.path.pop(0)
BRANCH = re.compile(r"s_branch|s_cbranch_\w+")


def regs(text):
    out = set()
    for kind, one, kind2, lo, hi in re.findall(r"\b([va])(\d+)\b|\b([va])\[(\d+):(\d+)\]", text):
        out |= {kind + one} if kind else {kind2 + str(i) for i in range(int(lo), int(hi) + 1)}
    return frozenset(out)


def kernels(asm):
    for m in re.finditer(r"^(_Z\S+):[^\n]*\n", asm, re.M):
        yield m.group(1), asm[m.end():asm.find(".Lfunc_end", m.end())]


def blocks_of(body):
    """[(label, [(mnemonic, operands, registers)])]"""
    out = [("", [])]
    for line in body.split("\n"):
        line = line.split(";")[0].strip()
        label = re.match(r"(\.LBB\w+):", line)
        if label:
            out.append((label.group(1), []))
        elif line and not line.startswith(".") and not line.endswith(":"):
            op, _, rest = line.partition(" ") if " " in line else line.partition("\t")
            out[-1][1].append((op.strip(), rest, regs(rest)))
    return out


def touched_in_flight(body):
    """Instructions that name a register of an LDS read before the wait that covers it (in order; other
    operations of the same counter take a place each), and the number of reads seen."""
    blocks = blocks_of(body)
    at = {label: i for i, (label, _) in enumerate(blocks)}
    bad, seen, work, reads = set(), set(), [(0, ())], 0
    while work:
        state = work.pop()
        if state in seen:
            continue
        seen.add(state)
        assert len(seen) < 100000
        i, flight = state[0], list(state[1])
        for op, rest, named in blocks[i][1]:
            if op == "s_waitcnt":
                n = re.search(r"lgkmcnt\((\d+)\)", rest)
                if n:
                    flight = flight[max(0, len(flight) - int(n.group(1))):] if int(n.group(1)) else []
                continue
            if named & frozenset().union(*flight):
                bad.add(f"{blocks[i][0]}: {op} {rest}")
            if op.startswith("ds_read"):
                flight.append(regs(rest.split(",")[0]))
                reads += 1
            elif op.startswith(("ds_", "s_load", "s_buffer_load")):
                flight.append(frozenset())
            if BRANCH.fullmatch(op):
                work.append((at[rest.strip()], tuple(flight)))
            if op in ("s_branch", "s_endpgm"):
                break
        else:
            if i + 1 < len(blocks):
                work.append((i + 1, tuple(flight)))
    return bad, reads


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm")

    def one(name):
        dst = str(out / (name + ".s"))
        subprocess.run([hipbuild.hipcc(), *hipbuild.HIPCC_FLAGS, "--cuda-device-only", "-S",
                        os.path.join(hipbuild.CSRC, name + ".hip"), "-o", dst], check=True, capture_output=True)
        return name, open(dst).read()
    with cf.ThreadPoolExecutor(3) as ex:
        return dict(ex.map(one, ("gemm", "head", "prefill")))


def test_no_register_of_a_read_in_flight_is_touched(assembly):
    want = {"gemm": ("gemm_tile_kernel", "gemm_dma_kernel"), "head": ("head_rows_kernel",),
            "prefill": ("attn_prefill_mfma_kernel",)}
    for name, asm in assembly.items():
        checked = set()
        for kernel, body in kernels(asm):
            if "ds_read" not in body:
                continue
            bad, reads = touched_in_flight(body)
            assert not bad, (kernel, sorted(bad)[:5])
            checked |= {w for w in want[name] if w in kernel and reads > 0}
        assert checked == set(want[name])


def test_the_walk_finds_a_missing_wait(assembly):
    """The last wait before the first product of each hand-waited kernel taken out (in the text)."""
    for name, kernel in (("gemm", "gemm_tile_kernel"), ("gemm", "gemm_dma_kernel"), ("head", "head_rows_kernel"),
                         ("prefill", "attn_prefill_mfma_kernel")):
        body = next(b for k, b in kernels(assembly[name]) if kernel in k)
        cut = body.index("v_mfma")
        at = body.rindex("lgkmcnt(", 0, cut) + len("lgkmcnt(")
        end = body.index(")", at)
        broken = body[:at] + "999" + body[end:]
        assert touched_in_flight(broken)[0], kernel
