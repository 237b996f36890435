"""The order of a block's stores and of the progress word that announces them, in the machine code of the built library.

The persistent closed loop publishes each block by one lane of one wave, after a barrier that closes the block; a
workgroup elsewhere then reads what all the waves of this one stored.  A workgroup barrier does not wait for the waves'
stores on this target, and the publishing wave's own wait covers its own stores only, so every wave has to wait for its
stores before that barrier.  A data-flow pass over the disassembly of the closed loop's kernels and of their block
functions checks it on every path.  Per wave it tracks
  pending   a store may be outstanding (set by a store, cleared by a wait for vmcnt 0),
  unsynced  a store may not be covered for another wave (set by a store; a barrier leaves it set only if the wave came to
            the barrier with a store pending).
Neither may hold where a block function (rc_luma, rc_chroma) returns, and unsynced may not where a word is stored in device
scope (the progress words; the abort flag), which is itself no data.  That is in recon_part, a function of its own in one
instance and inlined into the kernel in the other.  Every function waits at its entry; a call of a block function leaves
both clear, since its returns are checked, one of recon_part leaves unsynced set."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "av1gpu_amd", "libav1mi.so")
OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin" + os.pathsep + os.environ.get("PATH", ""))
STORE = re.compile(r"(global|flat|buffer)_(store|atomic)")
INSN = re.compile(r"^\s+(\S+)(.*?)\s*// ([0-9A-F]+):")
TARGET = re.compile(r"<(\S+?)(?:\+0x([0-9a-f]+))?>\s*$")


def code_objects():
    """The gfx950 code objects bundled in the library."""
    data, magic, at, out = open(LIB, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0, []
    while (at := data.find(magic, at)) >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24:p + 24 + tl]:
                out.append(data[at + off:at + off + size])
            p += 24 + tl
        at += 1
    return out


def functions(text):
    """name -> [(address, mnemonic, operands, branch target or None)] of the closed loop's kernels and block functions"""
    out, name, body = {}, None, None
    for line in text.splitlines():
        if line.endswith(">:"):
            start, name = line.split()[0], line.split("<", 1)[1][:-2]
            body = out.setdefault(name, []) if re.search(r"rc_(wide|narrow).*(rc_luma|rc_chroma|recon_part|k_recon_queue)I", name) else None
            base = int(start, 16)
        elif body is not None and (m := INSN.match(line)):
            t = TARGET.search(line) if m[1].startswith(("s_branch", "s_cbranch")) else None
            assert t is None or t[1] == name
            body.append((int(m[3], 16), m[1], m[2], base + int(t[2] or "0", 16) if t else None))
    return out


def step(state, op, args, parts):
    pending, unsynced = state
    if op == "s_barrier":
        unsynced = pending
    elif op == "s_waitcnt" and "vmcnt(0)" in args:
        pending = False
    elif op.startswith("s_swappc"):
        pending, unsynced = False, parts
    elif STORE.match(op) and not ("sc1" in args and "_store_" in op):
        pending = unsynced = True
    return pending, unsynced


def faults(body, returns=True, parts=False):
    """Addresses where a wave returns (if returns are to be checked), or stores a device-scope word, with stores that
    another wave may not see.  parts: the calls are of recon_part."""
    index = {a: i for i, (a, _, _, _) in enumerate(body)}
    seen, work, bad = {0: (False, False)}, [0], set()
    while work:
        i = work.pop()
        state = seen[i]
        while True:
            addr, op, args, target = body[i]
            if returns and op.startswith("s_setpc") and any(state) or "_store_" in op and "sc1" in args and state[1]:
                bad.add(addr)
            state = step(state, op, args, parts)
            nxt = [index[target]] if target is not None else []
            if not (op.startswith("s_setpc") or op in ("s_endpgm", "s_branch")):
                nxt.append(i + 1)
            go = []
            for j in nxt:
                new = tuple(a or b for a, b in zip(seen.get(j, (False, False)), state))
                if j not in seen or new != seen[j]:
                    seen[j] = new
                    go.append(j)
            if not go:
                break
            work += go[1:]
            i, state = go[0], seen[go[0]]
    return bad


@pytest.fixture(scope="module")
def code():
    assert OBJDUMP, "llvm-objdump of the ROCm toolchain"
    out = {}
    for k, co in enumerate(code_objects()):
        if b"k_recon_queue" not in co:
            continue
        path = os.path.join("/tmp", "publish_order_%d_%d.co" % (os.getpid(), k))
        with open(path, "wb") as f:
            f.write(co)
        try:
            out.update(functions(subprocess.run([OBJDUMP, "-d", path], check=True, capture_output=True, text=True).stdout))
        finally:
            os.remove(path)
    return out


@pytest.mark.parametrize("instance", ["rc_wide", "rc_narrow"])
@pytest.mark.parametrize("kind,count", [("rc_luma", 2 * 19), ("rc_chroma", 2 * 14)])
def test_a_block_ends_with_its_stores_complete(code, instance, kind, count):
    fns = {n: b for n, b in code.items() if instance in n and kind + "I" in n}
    assert len(fns) == count   # 8 and 16 bits per sample, every tx size
    for name, body in fns.items():
        ops = [op for _, op, _, _ in body]
        assert "s_barrier" in ops and any(STORE.match(op) for op in ops) and any(op.startswith("s_setpc") for op in ops)
        assert not faults(body), name


@pytest.mark.parametrize("instance", ["rc_wide", "rc_narrow"])
def test_a_block_is_published_after_its_stores(code, instance):
    kernels = {n: b for n, b in code.items() if instance in n and "k_recon_queueI" in n}
    parts = {n: b for n, b in code.items() if instance in n and "recon_partI" in n}
    assert len(kernels) == 2 and len(parts) in (0, 4)   # 8 and 16 bits per sample; luma and chroma
    words = [args for b in [*kernels.values(), *parts.values()] for _, op, args, _ in b if "_store_" in op and "sc1" in args]
    assert len(words) >= 2 * 3                          # luma block, chroma block, end of item
    for name, body in {**kernels, **parts}.items():
        assert not faults(body, returns=False, parts=bool(parts) and name in kernels), name


def test_every_function_waits_at_its_entry(code):
    for name, body in code.items():
        if "k_recon_queueI" not in name:
            entry = next(i for i, (_, op, args, _) in enumerate(body) if op == "s_waitcnt" and "vmcnt(0)" in args)
            assert not any(STORE.match(op) or op == "s_barrier" for _, op, _, _ in body[:entry]), name


def test_the_pass_finds_a_missing_wait():
    """On a made-up block: a store, a barrier and the word, with and without the wait, and with a wait on one path only."""
    def run(*ops):
        return bool(faults([(4 * k, op, args, t) for k, (op, args, t) in enumerate(ops)]))
    st, bar, word, end = ("global_store_dword", "v[0:1], v2, off", None), ("s_barrier", "", None), ("global_store_dword", "v0, v1 sc1", None), ("s_endpgm", "", None)
    wait = ("s_waitcnt", "vmcnt(0) lgkmcnt(0)", None)
    assert run(st, bar, word, end) and run(st, bar, wait, word, end) and run(st, wait, word, end)
    assert not run(st, wait, bar, word, end)
    assert run(st, ("s_cbranch_execz", "", 12), wait, bar, word, end)
    assert not run(("s_cbranch_execz", "", 8), st, wait, bar, word, end)
    assert run(st, bar, ("s_setpc_b64", "s[30:31]", None)) and run(bar, st, ("s_setpc_b64", "s[30:31]", None))
    assert not run(st, wait, bar, ("s_setpc_b64", "s[30:31]", None))
