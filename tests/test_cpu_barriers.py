"""A workgroup barrier does not wait for LDS stores by itself: every kernel of the built library waits for its own in front of each barrier, on every path.
(A raw barrier that forgets to lets another wave read, or store over, what is still under way; no run shows it reliably.)"""
import bisect
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "candle_vllm_amd", "libmi355vllm.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
CLEAN = -1


# function heads, and of the instructions those that the check looks at
LINE = re.compile(r"^(?:[0-9a-f]+ <([^>]+)>:|\t(ds_\S+|s_waitcnt|s_barrier|s_c?branch\S*|s_endpgm|s_load\S+|s_buffer_load\S+) *(.*?) *// ([0-9A-F]+):)", re.M)


def kernels(listing):
    """(name, [(address, instruction, operands)]) of every function of a listing"""
    name, body = None, []
    for m in LINE.finditer(listing):
        if m.group(1):
            if name:
                yield name, body
            name, body = m.group(1), []
        else:
            body.append((int(m.group(4), 16), m.group(2), m.group(3)))
    if name:
        yield name, body


def late_barriers(body):
    """addresses of the barriers that some path reaches with an LDS store under way.  A path's state: how many operations of the LDS counter it has issued from its
    last store on (CLEAN: the store is done) -- s_waitcnt lgkmcnt(n) leaves at most n of them, the oldest go first"""
    at = [ins[0] for ins in body]
    seen, work, late = [None] * len(body), [(0, CLEAN)], set()

    def worse(new, old):
        return old is None or (new != CLEAN and (old == CLEAN or new < old))
    while work:
        i, s = work.pop()
        while i < len(body) and worse(s, seen[i]):
            seen[i] = s
            addr, op, arg = body[i]
            if op.startswith(("ds_write", "ds_store", "ds_add")):
                s = 1
            elif op.startswith(("ds_", "s_load", "s_buffer_load")):
                s += s != CLEAN
            elif op == "s_waitcnt":
                left = re.search(r"lgkmcnt\((\d+)\)", arg)
                if arg in ("0", "0x0") or (left and s != CLEAN and int(left.group(1)) < s):
                    s = CLEAN
            elif op == "s_barrier" and s != CLEAN:
                late.add(addr)
            if op == "s_endpgm":
                break
            if op == "s_branch" or op.startswith("s_cbranch"):
                words = int(arg.split()[0])
                work.append((bisect.bisect_left(at, addr + 4 + 4 * (words - 65536 if words >= 32768 else words)), s))
                if op == "s_branch":
                    break
            i += 1
    return late


def test_the_check_itself():
    def run(*ops):
        return late_barriers([(4 * i, *op.partition(" ")[::2]) for i, op in enumerate(ops)])
    assert run("ds_write_b32 v0, v1", "s_barrier", "s_endpgm") == {4}
    assert not run("ds_write_b32 v0, v1", "s_waitcnt lgkmcnt(0)", "s_barrier", "s_endpgm")
    assert not run("ds_write_b32 v0, v1", "ds_read_b32 v2, v3", "s_waitcnt lgkmcnt(1)", "s_barrier", "s_endpgm")
    assert run("ds_write_b32 v0, v1", "s_waitcnt vmcnt(0)", "s_barrier", "s_endpgm") == {8}
    # a loop that waits in front of its barrier and stores behind it, and an exit that does not wait
    assert run("s_waitcnt lgkmcnt(0)", "s_barrier", "ds_write_b32 v0, v1", "s_cbranch_scc1 65532", "s_barrier", "s_endpgm") == {16}


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and ROCm's llvm-objdump")
def test_lds_stores_are_waited_for_in_front_of_every_barrier(tmp_path):
    copy = shutil.copy(LIB, tmp_path / "lib.so")                      # (the code objects are written next to it)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, stdout=subprocess.DEVNULL)
    found, late = 0, {}
    for obj in sorted(tmp_path.glob("lib.so.*gfx950")):
        with open(tmp_path / "listing", "w+b") as f:
            subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", obj], check=True, stdout=f)
        for name, body in kernels((tmp_path / "listing").read_text()):
            found += 1
            bad = late_barriers(body)
            if bad:
                late[name] = sorted(map(hex, bad))
    assert found > 100 and not late, late
