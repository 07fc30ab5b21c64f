"""The wait states between a matrix instruction and the first other instruction that touches its
result, in the disassembly of this repository's own device code, over every path of the control
flow.  hipcc counts them along some paths only where matrix instructions stand under branches
(csrc/mf_solve16.hip, mma_done); a path that is short of them reads the last result register early."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "cliquetrees.jl_amd", "libmfhip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

# wait states before another instruction may read or write the result: 16 and 8 passes and two
NEED = {"f64_16x16x4": 18, "f32_16x16x4": 10}


def _regs(text):
    out = set()
    for f, a, b in re.findall(r"\b([va])\[(\d+):(\d+)\]", text):
        out |= {f + str(i) for i in range(int(a), int(b) + 1)}
    out |= {f + n for f, n in re.findall(r"\b([va])(\d+)\b", text)}
    return out


def parse(listing):
    """[(address, mnemonic, operands)] of an objdump listing."""
    ins = []
    for line in listing.splitlines():
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+):", line)
        if m:
            ins.append((int(m.group(3), 16), m.group(1), m.group(2)))
    return ins


def short_paths(ins):
    """(address of the matrix instruction, address of the early one, wait states between).

    An instruction is early that reads the result, or (but for loads, whose data comes later than
    that) writes it.  Where a branch is taken because EXEC is 0, vector instructions do nothing
    until EXEC is written."""
    at = {a: i for i, (a, _, _) in enumerate(ins)}

    def following(i, off):
        a, op, args = ins[i]
        if op in ("s_endpgm", "s_setpc_b64"):
            return []
        if args.startswith("exec") or "saveexec" in op:
            off = False
        if op.startswith("s_cbranch") or op == "s_branch":
            d = int(args.split()[0])
            t = at.get(a + 4 + 4 * (d - 65536 if d >= 32768 else d))
            assert t is not None, (hex(a), op, args)
            taken = (t, off or op == "s_cbranch_execz")
            return [taken] if op == "s_branch" else [(i + 1, off), taken]
        return [(i + 1, off)]

    known = {}

    def touched(j):
        """Registers that instruction j may be early for, and those whose old value it ends."""
        if j not in known:
            _, op, args = ins[j]
            first, _, rest = args.partition(", ")
            load = "load" in op or op.startswith("ds_read") or "bpermute" in op
            known[j] = (_regs(rest), _regs(first)) if load else (_regs(args), set())
        return known[j]

    bad = []
    for i, (a, op, args) in enumerate(ins):
        if not op.startswith("v_mfma"):
            continue
        need = [v for k, v in NEED.items() if k in op]
        assert need, op
        best = {}
        todo = [(j, 0, frozenset(_regs(args.split(", ")[0])), off) for j, off in following(i, False)]
        while todo:
            j, waited, live, off = todo.pop()
            if j >= len(ins) or waited >= need[0] or not live or best.get((j, live, off), 99) <= waited:
                continue
            best[j, live, off] = waited
            b, o, x = ins[j]
            states = 1
            if o.startswith("v_mfma"):
                # sums that go on are checked from there; a new result ends the old one
                rest = live - _regs(x.split(", ")[0])
                if rest != live:
                    continue
                states = need[0] - 2
            elif o == "s_nop":
                states = int(x, 0) + 1
            elif not off:
                early, ends = touched(j)
                if early & live:
                    bad.append((a, b, waited))
                    break
                live = live - ends
            todo += [(k, waited + states, live, f) for k, f in following(j, off)]
    return bad


def test_checker():
    """A branch around the second of two products: its path reads the first one's sum at once."""
    text = """
	v_mfma_f64_16x16x4_f64 v[0:7], v[8:9], v[10:11], v[0:7]    // 000000000100: 00000000 00000000
	s_cbranch_scc1 2                                           // 000000000108: 00000000
	v_mfma_f64_16x16x4_f64 v[20:27], v[8:9], v[10:11], v[20:27]// 00000000010C: 00000000 00000000
	s_nop {}                                                   // 000000000114: 00000000
	v_mov_b32_e32 v30, v7                                      // 000000000118: 00000000
	s_endpgm                                                   // 00000000011C: 00000000
"""
    assert short_paths(parse(text.format(0))) == [(0x100, 0x118, 2)]
    assert short_paths(parse(text.format(15))) == [(0x100, 0x118, 17)]
    ok = text.format(15).replace("v_mov_b32_e32 v30, v7", "v_mov_b32_e32 v30, v8")
    assert short_paths(parse(ok)) == []


def test_library(tmp_path):
    if not (os.path.exists(OBJDUMP) and os.path.exists(LIB)):
        pytest.skip("no llvm-objdump or no built library")
    link = tmp_path / "lib.so"
    link.symlink_to(LIB)
    subprocess.run([OBJDUMP, "--offloading", str(link)], check=True, capture_output=True, cwd=tmp_path)
    count = 0
    for name in sorted(os.listdir(tmp_path)):
        if "amdgcn" not in name:
            continue
        text = subprocess.run([OBJDUMP, "-d", str(tmp_path / name)], check=True, capture_output=True, text=True).stdout
        ins = parse(text)
        count += sum(op.startswith("v_mfma") for _, op, _ in ins)
        bad = short_paths(ins)
        assert not bad, (name, [(hex(a), hex(b), w) for a, b, w in bad[:8]])
    assert count > 1000
