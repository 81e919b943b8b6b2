"""No register of an LDS read is touched before the wait that covers it, in the built kernels.

csrc/attn.hip and csrc/dense.hip issue LDS reads through inline asm and wait for some of them in a later statement.  In between the compiler
believes the destinations are written already; a copy, a spill or a reuse of such a register there would go wrong without a word.
This test disassembles the kernels of the built library and follows every path through them: LDS operations finish in order, so a
read with n later LDS operations is done behind `s_waitcnt lgkmcnt(m)` with m <= n (a scalar load under way shares the counter
and only makes the wait longer)."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "spargeattn_amd", "libspargeattn_amd.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])(?![\w(])")
LGKM = re.compile(r"lgkmcnt\((\d+)\)")
BRANCH = re.compile(r"^(s_branch|s_cbranch_\w+)$")
TARGET = re.compile(r"<[^>]*?(?:\+0x([0-9a-f]+))?>\s*$")


def code_objects(path):
    """The gfx950 code objects of the library's offload bundles."""
    data, magic = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        entries, pos = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(entries):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            if size and b"gfx950" in data[pos + 24:pos + 24 + n]:
                yield data[at + off:at + off + size]
            pos += 24 + n
        at = data.find(magic, at + len(magic))


def registers(text):
    out = set()
    for kind, one, lo, hi in REG.findall(text):
        out.update((kind, i) for i in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
    return out


def functions(asm):
    """name -> [(address, mnemonic, operands, branch target or None)] of llvm-objdump's text."""
    name, base, out = None, 0, {}
    for line in asm.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:$", line)
        if head:
            base, name = int(head[1], 16), head[2]
            out[name] = []
        elif name is not None and "//" in line:
            text, _, tail = line.partition("//")
            mnemonic, _, ops = text.strip().partition(" ")
            target = None
            if BRANCH.match(mnemonic):
                target = base + int(TARGET.search(tail)[1] or "0", 16)
            out[name].append((int(tail.split(":")[0], 16), mnemonic, ops, target))
    return out


def violations(code):
    """Instructions that name a register of an LDS read in flight.  code: one function as `functions` gives it."""
    index = {addr: i for i, (addr, _, _, _) in enumerate(code)}
    starts = {0} | {index[t] for _, _, _, t in code if t is not None} | {i + 1 for i, c in enumerate(code) if c[3] is not None}
    regs = [registers(ops) for _, _, ops, _ in code]
    state_at, work, bad = {0: {}}, [0], set()
    while work:
        i = work.pop()
        flight = dict(state_at[i])                        # register -> LDS operations behind its read
        while True:
            addr, op, ops, target = code[i]
            if op == "s_waitcnt":
                m = LGKM.search(ops)
                if m:
                    flight = {r: n for r, n in flight.items() if n < int(m[1])}
            elif flight and not regs[i].isdisjoint(flight):
                bad.add((hex(addr), op, ops))
            assert not op.startswith("flat_"), "counts as an LDS operation, too"
            if op.startswith("ds_"):
                flight = {r: n + 1 for r, n in flight.items()}
                if op.startswith(("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle")) or "_rtn" in op:
                    flight.update((r, 0) for r in registers(ops.split(",")[0]))
            follow = [] if op in ("s_endpgm", "s_branch") else [i + 1]
            if target is not None:
                follow.append(index[target])
            if len(follow) == 1 and follow[0] == i + 1 and i + 1 not in starts:
                i += 1
                continue
            for j in follow:
                if j >= len(code):
                    continue
                old = state_at.get(j)
                new = dict(flight) if old is None else {r: min(old.get(r, 99), flight.get(r, 99)) for r in old.keys() | flight.keys()}
                if new != old:
                    state_at[j] = new
                    work.append(j)
            break
    return bad


@pytest.fixture(scope="module")
def kernels():
    if not (os.path.exists(LIB) and os.path.exists(OBJDUMP)):
        pytest.skip("no built library or no llvm-objdump")
    out = {}
    for i, obj in enumerate(code_objects(LIB)):
        if b"block_sparse_attn_kernel" in obj or b"dense_attn_f16_kernel" in obj:
            r = subprocess.run([OBJDUMP, "-d", "-"], input=obj, capture_output=True)
            assert r.returncode == 0, r.stderr[-500:]
            out.update({k: v for k, v in functions(r.stdout.decode()).items() if "attn" in k or "row_maxima" in k})
    return out


def test_every_read_is_waited_for_first(kernels):
    attn = [k for k in kernels if "block_sparse_attn_kernel" in k]
    assert len(attn) >= 60 and all(any(name in k for k in kernels) for name in ("few_rows_attn_kernel", "row_maxima_kernel", "dense_attn_f16_kernel"))
    for name, code in kernels.items():
        assert sum(op == "ds_read_b128" for _, op, _, _ in code) > 0, name
        assert not violations(code), name


def _code(text):
    lines = [l.strip() for l in text.strip().splitlines()]
    labels, ins = {}, []
    for l in lines:
        if l.endswith(":"):
            labels[l[:-1]] = len(ins)
        else:
            ins.append(l.partition(" ")[::2])
    return [(4 * i, op, ops, 4 * labels[ops] if BRANCH.match(op) else None) for i, (op, ops) in enumerate(ins)]


@pytest.mark.parametrize("text,count", [
    ("ds_read_b128 v[0:3], v8\ns_waitcnt lgkmcnt(0)\nv_mov_b32_e32 v9, v3\ns_endpgm", 0),
    ("ds_read_b128 v[0:3], v8\nv_mov_b32_e32 v9, v3\ns_waitcnt lgkmcnt(0)\ns_endpgm", 1),
    ("ds_read_b128 v[0:3], v8\nv_mov_b32_e32 v2, v9\ns_endpgm", 1),
    ("ds_read_b128 v[0:3], v8\nds_read_b128 v[4:7], v8\ns_waitcnt lgkmcnt(1)\nv_mov_b32_e32 v9, v3\ns_endpgm", 0),
    ("ds_read_b128 v[0:3], v8\nds_read_b128 v[4:7], v8\ns_waitcnt vmcnt(0) lgkmcnt(1)\nv_mov_b32_e32 v9, v4\ns_endpgm", 1),
    ("ds_read_b128 v[0:3], v8\ns_waitcnt vmcnt(0)\nv_mov_b32_e32 v9, v3\ns_endpgm", 1),
    # in flight on one of two paths, and round a loop
    ("s_cbranch_scc1 a\nds_read_b32 v0, v8\na:\nv_mov_b32_e32 v9, v0\ns_endpgm", 1),
    ("ds_read_b32 v0, v8\ns_cbranch_scc1 a\ns_waitcnt lgkmcnt(0)\na:\nv_mov_b32_e32 v9, v0\ns_endpgm", 1),
    ("a:\nv_mov_b32_e32 v9, v0\nds_read_b32 v0, v8\ns_cbranch_scc1 a\ns_endpgm", 2),
    ("a:\ns_waitcnt lgkmcnt(0)\nv_mov_b32_e32 v9, v0\nds_read_b32 v0, v8\ns_cbranch_scc1 a\ns_endpgm", 0),
    ("ds_write_b128 v8, v[0:3]\nv_mov_b32_e32 v0, v9\ns_endpgm", 0)])
def test_the_check_itself(text, count):
    assert len(violations(_code(text))) == count
