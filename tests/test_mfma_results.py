"""Matrix products' results are not read before they are there.

The hardware does not hold back a vector or memory instruction that uses an
MFMA's result too early: the instructions between have to take up enough issue
states (the product's passes + 3, one more on gfx950 from 4 passes on).  The
compiler pads to that, but counts every s_waitcnt as a state, and by what was
seen one that is already satisfied takes none.  So the states are counted here without waits and
barriers, over every path, in the assembly of each source that has products,
built with the library's own flags.
"""
import re
import subprocess

import pytest

from cpubrrr_amd import build as B

# passes of the products in use; f8f6f4 with an fp8 operand
PASSES = {
    "v_mfma_scale_f32_32x32x64_f8f6f4": 16,
    "v_mfma_scale_f32_16x16x128_f8f6f4": 8,
    "v_mfma_i32_32x32x32_i8": 8,
    "v_mfma_i32_32x32x16_i8": 8,
}
REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")


def regs(text):
    out = set()
    for f, one, lo, hi in REG.findall(text):
        out |= {(f, i) for i in (range(int(lo), int(hi) + 1) if lo else (int(one),))}
    return out


def parse(asm):
    """{kernel: (instructions [(opcode, operands)], label -> index)}"""
    kernels, cur = {}, None
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        if m := re.match(r"(_Z\w+):", line):
            cur = kernels[m[1]] = ([], {})
        elif cur is None or not line or line.startswith("//"):
            continue
        elif line.startswith(".Lfunc_end"):
            cur = None
        elif m := re.match(r"(\.\w+):", line):
            cur[1][m[1]] = len(cur[0])
        elif not line.startswith("."):
            op, _, rest = line.partition(" ")
            cur[0].append((op.split("\t")[0], line[len(op.split("\t")[0]):]))
    return {k: v for k, v in kernels.items() if any(op.startswith("v_mfma") for op, _ in v[0])}


def states(op, rest):
    if op == "s_nop":
        return int(rest, 0) + 1
    return 0 if op.startswith("s_waitcnt") or op in ("s_barrier", "s_setprio") else 1


def too_early(ins, labels):
    """(product, use, states between, states needed) of every use that comes too early"""
    found = []
    for p, (op, rest) in enumerate(ins):
        if not op.startswith("v_mfma"):
            continue
        need = PASSES[op] + 4
        dst = regs(rest.split(",")[0])
        todo, seen = [(p + 1, 0)], {}
        while todo:
            i, n = todo.pop()
            while n < need and seen.get(i, need) > n:
                seen[i] = n
                o, r = ins[i]
                if o == "s_endpgm":
                    break
                if not o.startswith(("s_", "v_mfma")) and regs(r) & dst:
                    found.append((f"{p}: {op}{rest}", f"{i}: {o}{r}", n, need))
                    break
                n += states(o, r)
                if o.startswith(("s_branch", "s_cbranch")):
                    todo.append((labels[r.strip()], n))
                    if o == "s_branch":
                        break
                i += 1
    return found


def assembly(source):
    cmd = [B.HIPCC, *B.COMMON, "-S", "--cuda-device-only", str(B.CSRC / source), "-o", "-"]
    return subprocess.run(cmd, check=True, stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True).stdout


@pytest.mark.parametrize("source", ["moe_mx.hip", "moe_grouped.hip", "moe_grouped_kq.hip"])
def test_results_are_there(source):
    kernels = parse(assembly(source))
    assert kernels
    bad = {k: too_early(*v) for k, v in kernels.items()}
    assert not any(bad.values()), "\n".join(f"{k}: {len(b)} uses too early, the first: {b[0]}" for k, b in bad.items() if b)


def test_other_sources_have_no_products():
    for s in set(B.SOURCES) - {"moe_mx.hip", "moe_grouped.hip", "moe_grouped_kq.hip"}:
        assert "__builtin_amdgcn_mfma" not in (B.CSRC / s).read_text()


def test_counting():
    d = "v_mfma_i32_32x32x32_i8"
    def early(*lines):
        asm = "_Zk:\n" + f"\t{d} v[0:15], v[20:23], v[24:27], 0\n" + "\n".join("\t" + l for l in lines) + "\n\ts_endpgm\n.Lfunc_end0:\n"
        return [(n, need) for _, _, n, need in too_early(*parse(asm)["_Zk"])]
    pad = ["v_mov_b32_e32 v30, v31"] * 11
    assert early(*pad, "v_mov_b32_e32 v30, v15") == [(11, 12)]
    assert early(*pad, "s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v30, v15") == [(11, 12)]
    assert early("s_nop 10", "s_add_i32 s0, s0, 1", "v_mov_b32_e32 v30, v15") == []
    assert early(*pad, "v_mov_b32_e32 v30, v16", "ds_write_b128 v40, v[12:15]") == []
    assert early("s_cbranch_scc1 .L1", *pad, "v_mov_b32_e32 v30, v31", ".L1:", "ds_write_b128 v40, v[12:15]") == [(1, 12)]
