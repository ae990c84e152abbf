"""Loads that write LDS by themselves, and sums that are parked there: the waits of the compiled kernels.

The tiles of vkl_gemm_wide.hip put their sums where the stages of their loads were.  A load that is still in flight then
writes over sums of any wave, and a wave can wait for its own loads only: so all of them have landed before the barrier
behind which the first sum is written.  No result shows a wait that is missing (the loads are late once in a great while),
so the instructions are followed along every branch instead."""
import os
import re
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vkllama_amd", "lib", "libvkllama_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def listing(tmp):
    """{kernel: [(address, opcode, operands)]} of the wide products' object"""
    at = os.path.join(tmp, "lib.so")
    os.symlink(LIB, at)
    subprocess.run([OBJDUMP, "--offloading", at], check=True, capture_output=True, cwd=tmp)
    for name in os.listdir(tmp):
        path = os.path.join(tmp, name)
        if "gfx950" not in name or b"gemm_mix_kernel" not in open(path, "rb").read():
            continue
        text = subprocess.run([OBJDUMP, "-d", path], check=True, capture_output=True, text=True).stdout
        kernels, now = {}, None
        for line in text.splitlines():
            head = re.match(r"[0-9a-f]+ <(\w+)>:", line)
            if head:
                now = kernels.setdefault(head.group(1), [])
            code = re.match(r"\s+(\w+)(.*?)\s*// ([0-9A-F]+): ([0-9A-F]{8})", line)
            if code:
                now.append((int(code.group(3), 16), code.group(1), code.group(2), int(code.group(4), 16)))
        return kernels
    raise AssertionError("no such object in " + LIB)


def follow(code):
    """Addresses at which LDS is written, or the wave ends, while loads into it may be in flight.

    Before each instruction: bit 0, loads of this wave may be in flight; bit 1, so they were at the last barrier, and those
    of other waves may be.  All waves run the same code, so one stands for the others."""
    index = {a: i for i, (a, *_) in enumerate(code)}
    state, todo, found = {0: {0}}, [(0, 0)], set()
    while todo:
        i, s = todo.pop()
        addr, op, rest, word = code[i]
        if op.startswith("global_load_lds"):
            s |= 1
        elif op == "s_waitcnt" and "vmcnt(0)" in rest:
            s &= ~1
        elif op == "s_barrier":
            s = 3 if s & 1 else 0
        elif (op.startswith("ds_write") and s) or (op == "s_endpgm" and s & 1):
            found.add(addr)
        nxt = []
        if op in ("s_branch",) or op.startswith("s_cbranch"):
            off = word & 0xffff
            nxt.append(index[addr + 4 + 4 * (off - 0x10000 if off & 0x8000 else off)])
        assert op not in ("s_setpc_b64", "s_swappc_b64")
        if op not in ("s_branch", "s_endpgm"):
            nxt.append(i + 1)
        for n in nxt:
            if s not in state.setdefault(n, set()):
                state[n].add(s)
                todo.append((n, s))
    return found


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and its disassembler")
def test_no_load_is_in_flight_where_sums_are_parked(tmp_path):
    kernels = {k: v for k, v in listing(str(tmp_path)).items() if "gemm_mix" in k or "gemm_wide" in k}
    loads = {k: sum(op.startswith("global_load_lds") for _, op, *_ in v) for k, v in kernels.items()}
    parks = {k: sum(op.startswith("ds_write") for _, op, *_ in v) for k, v in kernels.items()}
    assert len(kernels) >= 15 and min(loads.values()) > 0 and min(parks.values()) > 0
    late = {k: sorted(map(hex, follow(v)))[:4] for k, v in kernels.items()}
    assert not any(late.values()), {k: v for k, v in late.items() if v}


def test_the_way_is_followed():
    """The four ways to go wrong, and the right one, by hand."""
    load, wait, some = ("global_load_lds_dwordx4", "", 0), ("s_waitcnt", "vmcnt(0)", 0), ("s_waitcnt", "vmcnt(2)", 0)
    barrier, write, end = ("s_barrier", "", 0), ("ds_write_b128", "", 0), ("s_endpgm", "", 0)

    def late(*ops):
        return bool(follow([(4 * i, *op) for i, op in enumerate(ops)]))
    assert not late(load, wait, barrier, write, end)
    assert late(load, barrier, wait, write, end)                   # its own loads only
    assert late(load, wait, load, barrier, wait, write, end)
    assert late(load, some, barrier, write, wait, end)
    assert late(load, some, end)
    assert late(load, ("s_cbranch_scc0", "", 1), wait, barrier, write, end)      # around the wait
    assert not late(load, wait, ("s_cbranch_scc0", "", 0xfffe), barrier, write, end)  # a loop
