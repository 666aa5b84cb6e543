"""CPU test of the GEMM kernels' waits, on the gfx950 code that the library holds.

The tiled GEMMs copy the activation from global memory to LDS and load the
weights into registers with instructions that share one counter (vmcnt), and
wait with a count: "all but the newest N".  N is the number of weight loads
issued after the copies, so it is right only if the compiler leaves the copies
before them.  A copy that sinks past a counted load is not waited for, and the
workgroup reads what the LDS held before: a race that results seldom show.

So the compiled kernels are read: over every path to an s_barrier, every copy
to LDS issued so far has been waited for."""
import os
import re
import shutil
import subprocess

import pytest

from arm_ai_amd import build

OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and os.path.exists(p)), None)
NAMES = [b"kq6kernelI", b"pair_kernelI", b"gemm8_kernelI"]
DONE = 1 << 20  # no copy outstanding

INSTR = re.compile(r"^\s+([a-z][a-z0-9_]+)(.*?)//\s*([0-9A-F]+):")
TARGET = re.compile(r"<.*\+0x([0-9a-f]+)>\s*$|<([^+>]*)>\s*$")


def functions(path):
    """{kernel name: [(address, mnemonic, operands, line)]} of an AMD code object."""
    out = subprocess.run([OBJDUMP, "-d", path], capture_output=True, text=True, check=True).stdout
    funcs, name, base = {}, None, 0
    for line in out.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:$", line)
        if head:
            name, base = head.group(2), int(head.group(1), 16)
            funcs[name] = (base, [])
            continue
        m = INSTR.match(line)
        if m and name:
            funcs[name][1].append((int(m.group(3), 16), m.group(1), m.group(2), line))
    return funcs


def after(state, op, args):
    """state: memory operations issued after the newest copy that may still be
    under way; the value after one more instruction."""
    if op == "s_waitcnt":
        m = re.search(r"vmcnt\((\d+)\)", args)
        # the newest N stay: the copy among them has `state` newer ones
        if m and state >= int(m.group(1)):
            return DONE
        return state
    if op.startswith(("buffer_", "global_", "flat_", "scratch_")) and not op.startswith(("buffer_wbl2", "buffer_inv")):
        if "lds" in args.split() or "_lds_" in op:
            return 0
        return state if state == DONE else min(state + 1, 64)
    return state


def unwaited_barriers(base, code):
    """Addresses of the barriers that a copy to LDS can reach under way."""
    index = {a: i for i, (a, *_r) in enumerate(code)}
    succ = []
    for i, (_a, op, _args, line) in enumerate(code):
        nxt = [i + 1] if i + 1 < len(code) else []
        if op == "s_endpgm":
            nxt = []
        elif op == "s_branch" or op.startswith("s_cbranch"):
            m = TARGET.search(line)
            assert m, line
            to = index[base + int(m.group(1) or "0", 16)]
            nxt = [to] if op == "s_branch" else nxt + [to]
        assert not op.startswith(("s_setpc", "s_swappc", "s_call")), line
        succ.append(nxt)
    state = [None] * len(code)
    state[0] = DONE
    work = [0]
    while work:
        i = work.pop()
        s = after(state[i], code[i][1], code[i][2])
        for j in succ[i]:
            if state[j] is None or s < state[j]:
                state[j] = s
                work.append(j)
    return [hex(a) for i, (a, op, *_r) in enumerate(code) if op == "s_barrier" and state[i] is not None and state[i] != DONE]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if OBJDUMP is None or not os.path.exists(build.LIB):
        pytest.skip("llvm-objdump or the built library is missing")
    work = tmp_path_factory.mktemp("code")
    lib = shutil.copy(build.LIB, work / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=work, capture_output=True, check=True)
    funcs = {}
    for f in sorted(work.iterdir()):
        if "amdgcn" in f.name and any(n in f.read_bytes() for n in NAMES):  # (the others are large)
            funcs.update(functions(str(f)))
    return funcs


# the K-quant tiles of every type, the pair of two weights, the Q8_0 tiles
@pytest.mark.parametrize("name,least", [("2kq6kernelI", 25), ("2kq11pair_kernelI", 2), ("12gemm8_kernelI", 1)])
def test_copies_are_waited_for(kernels, name, least):
    found = {n: c for n, c in kernels.items() if name in n}
    assert len(found) >= least
    bad = {}
    for n, (base, code) in found.items():
        assert any("lds" in args.split() for _a, _op, args, _l in code), n
        at = unwaited_barriers(base, code)
        if at:
            bad[n] = at
    assert not bad, bad
