"""No kernel uses a register whose load is still in flight.

The GEMM kernels read LDS with inline asm, which the compiler takes as complete at once, and wait
by hand. A wait that comes too late for one use (or for a copy that the compiler puts at a branch or
loop edge) gives wrong results only when the read happens to be slow, which no run shows reliably.
So this walks the built library's own device code: along every path of every kernel, the loads
whose completion no s_waitcnt has established, and any instruction that names one of their
destination registers. Both counters are followed; LDS operations complete in order, vector-memory
operations too, and scalar loads, which share the LDS counter but complete in any order, are
counted as done (the remaining count then stands for LDS operations, which is the worse case).
"""
import os
import re
import shutil
import subprocess

import pytest

from justgoal_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
pytestmark = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs llvm-objdump")

# every kernel family of the library
FAMILIES = ("route_kernel", "route_permute_kernel", "permute_kernel", "combine_kernel",
            "quant_act_kernel", "gemm1_stream_kernel", "gemm1_tile_kernel", "gemm1_big_kernel",
            "gemm2_stream_kernel", "gemm2_tile_kernel", "gemm2_token_kernel", "gemm2_wide_kernel",
            "gemm2_big_kernel")

REGS = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])(?!\w)")
LINE = re.compile(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<[^>+]*(?:\+0x([0-9a-f]+))?>)?\s*$")
LDS_LOADS = ("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle")
LGKM_MAX, VM_MAX = 15, 63  # what the counters hold: an instruction past that waits to be issued


def registers(operands):
    out = set()
    for kind, one, lo, hi in REGS.findall(operands):
        out.update((kind, i) for i in range(int(one or lo), int(one or hi) + 1))
    return frozenset(out)


def parse(text):
    """llvm-objdump -d text -> {symbol: [(address, mnemonic, operands, branch target or None)]}"""
    kernels, code, base = {}, None, 0
    for line in text.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.*)>:", line)
        if head:
            base, code = int(head[1], 16), kernels.setdefault(head[2], [])
            continue
        m = LINE.match(line)
        if m is None:
            assert code is None or not line.strip() or line.strip() == "...", line
            continue
        branch = m[1].startswith(("s_cbranch", "s_branch"))
        code.append((int(m[3], 16), m[1], m[2], base + int(m[4] or "0", 16) if branch else None))
    return kernels


def merge(a, b):
    """Union of two states; operations are matched by how many were issued after them."""
    if a is None:
        return b
    out = []
    for x, y in zip(a, b):
        n = max(len(x), len(y))
        x = (frozenset(),) * (n - len(x)) + x
        y = (frozenset(),) * (n - len(y)) + y
        out.append(tuple(p | q for p, q in zip(x, y)))
    return tuple(out)


def step(state, op, operands):
    """State after the instruction, and the registers in flight that it names."""
    lgkm, vm = state
    if op == "s_waitcnt":
        def left(ops, name):
            m = re.search(name + r"\((\d+)\)", operands)
            return ops[max(0, len(ops) - int(m[1])):] if m else ops
        return (left(lgkm, r"\blgkmcnt"), left(vm, r"\bvmcnt")), frozenset()
    used = registers(operands)
    bad = used & frozenset().union(*lgkm, *vm)
    first = registers(operands.split(",")[0])
    if op.startswith("ds_"):
        dest = first if op.startswith(LDS_LOADS) or "_rtn" in op else frozenset()
        lgkm = (lgkm + (dest,))[-LGKM_MAX:]
    elif op.startswith(("buffer_", "global_", "scratch_", "flat_")):
        to_lds = re.search(r"\blds\b", operands) is not None
        dest = first if "_load" in op and not to_lds else frozenset()
        vm = (vm + (dest,))[-VM_MAX:]
    return (lgkm, vm), bad


def uses_in_flight(code):
    """[(address, instruction)] that name a register whose load may still be in flight."""
    index = {ins[0]: i for i, ins in enumerate(code)}
    states = [None] * len(code)
    states[0] = ((), ())
    work, bad = [0], {}
    while work:
        i = work.pop()
        _, op, operands, target = code[i]
        after, hit = step(states[i], op, operands)
        if hit:
            bad[code[i][0]] = f"{op} {operands}"
        if op == "s_endpgm":
            continue
        succ = [] if target is None else [index[target]]
        if op != "s_branch" and i + 1 < len(code):
            succ.append(i + 1)
        for n in succ:
            merged = merge(states[n], after)
            if merged != states[n]:
                states[n] = merged
                work.append(n)
    return sorted(bad.items())


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(build.LIB_PATH):
        build.build()
    tmp = tmp_path_factory.mktemp("isa")
    lib = shutil.copy(build.LIB_PATH, tmp / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True, cwd=tmp)
    out = {}
    for f in sorted(tmp.glob(f"lib.so.*{build.ARCH}")):
        text = subprocess.run([OBJDUMP, "-d", str(f)], check=True, capture_output=True, text=True)
        out.update(parse(text.stdout))
    return out


def test_every_kernel_is_walked(kernels):
    assert all(re.search(rf"\d({'|'.join(FAMILIES)})[IE]", k) for k in kernels)


@pytest.mark.parametrize("name", FAMILIES)
def test_no_register_is_used_while_its_load_is_in_flight(kernels, name):
    mine = {k: v for k, v in kernels.items() if re.search(rf"\d{name}[IE]", k)}
    assert mine
    for symbol, code in mine.items():
        assert not uses_in_flight(code), symbol


def listing(*instructions):
    """Assembly lines in objdump's form, 4 bytes each; '@n' as the operand of a branch is its
    target's index."""
    out = ["0000000000001000 <k>:"]
    for i, text in enumerate(instructions):
        text, _, target = text.partition("@")
        mark = f" <k+0x{4 * int(target):x}>" if target else ""
        out.append(f"\t{text}  // {0x1000 + 4 * i:012X}: BF800000{mark}")
    return parse("\n".join(out))["k"]


@pytest.mark.parametrize("lines,bad", [
    (("ds_read_b32 v1, v2", "s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v3, v1", "s_endpgm"), []),
    (("ds_read_b32 v1, v2", "v_mov_b32_e32 v3, v1", "s_waitcnt lgkmcnt(0)", "s_endpgm"), [1]),
    # a copy at a loop's head of what the loop's end reads
    (("v_mov_b32_e32 v3, v1", "s_waitcnt lgkmcnt(0)", "ds_read_b128 v[0:3], v9",
      "s_cbranch_scc1 65532 @0", "s_endpgm"), [0]),
    # counted waits: the older read is done, the younger is not
    (("ds_read_b32 v1, v9", "ds_read_b32 v2, v9", "s_waitcnt lgkmcnt(1)", "v_add_u32_e32 v4, v1, v1",
      "v_add_u32_e32 v4, v2, v2", "s_endpgm"), [4]),
    # a write to the register of a load in flight; a DMA into LDS has no register of its own
    (("buffer_load_dword v1, v2, s[0:3], 0 offen", "v_mov_b32_e32 v1, 0", "s_endpgm"), [1]),
    (("buffer_load_dword v1, s[0:3], 0 offen lds", "v_mov_b32_e32 v1, 0", "s_endpgm"), []),
    # one of two paths waits
    (("ds_read_b32 v1, v2", "s_cbranch_scc0 1 @3", "s_waitcnt lgkmcnt(0)", "v_mov_b32_e32 v3, v1",
      "s_endpgm"), [3]),
])
def test_walk_finds_planted_uses(lines, bad):
    got = [(a - 0x1000) // 4 for a, _ in uses_in_flight(listing(*lines))]
    assert got == bad
