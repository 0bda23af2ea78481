"""The tiled GEMM's MFMAs are inline assembly: the compiler does not know how long their results stay in the matrix pipe and
puts no wait states before an instruction that reads or overwrites an accumulator.  The body of the K loops ends in a wait of its
own (s_nop 7: what the compiler keeps behind the same MFMA as a builtin); here the built kernels are followed through every branch: only another MFMA touches an accumulator before it."""
import re
import shutil
import struct
import subprocess

import pytest

from mi355x_qlinear import capi

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:/opt/rocm/lib/llvm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 code objects of the bundles in a shared library: magic, count, then (offset, size, triple) each."""
    for start in (m.start() for m in re.finditer(MAGIC, data)):
        at = start + len(MAGIC)
        count, = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in triple and size:
                yield data[start + offset:start + offset + size]


def _kernels(path):
    """(name, [(address, instruction, branch target or None)]) of every gemm_tiled_kernel of a code object."""
    text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
    for block in text.split("\n\n"):
        head = re.match(r"([0-9a-f]+) <(\S*gemm_tiled_kernel\S*)>:", block.strip())
        if not head:
            continue
        base, body = int(head[1], 16), []
        for m in re.finditer(r"^\t(\w+)([^\n]*?)\s*// ([0-9A-F]+):([^\n]*)$", block, re.M):
            to = re.search(r"<\S+?\+0x([0-9a-f]+)>", m[4])
            body.append((int(m[3], 16), m[1] + m[2], base + int(to[1], 16) if to else None))
        yield head[2], body


def _accumulators(operands):
    """Bit mask of the AGPRs in a list of operands."""
    mask = 0
    for m in re.finditer(r"\ba(?:\[(\d+):(\d+)\]|(\d+)\b)", operands):
        lo, hi = (int(m[3]),) * 2 if m[3] else (int(m[1]), int(m[2]))
        mask |= (1 << hi + 1) - (1 << lo)
    return mask


def _touched_in_flight(body):
    """Instructions that touch an AGPR which, on some path, is the result of an MFMA with no wait behind it."""
    index = {a: i for i, (a, _, _) in enumerate(body)}
    ops = [t.split(None, 1) + [""] for _, t, _ in body]
    wait = [o[0] == "s_nop" and int(o[1], 0) >= 7 for o in ops]
    starts, use = [0] * len(body), [0] * len(body)
    for i, o in enumerate(ops):
        if o[0].startswith("v_mfma"):
            starts[i] = _accumulators(o[1].split(",")[0])
        else:
            use[i] = _accumulators(o[1])
    state, todo = {0: 0}, [0]
    while todo:
        i = todo.pop()
        after = 0 if wait[i] else state[i] | starts[i]
        op, to = ops[i][0], body[i][2]
        assert to is not None or not re.match(r"s_c?branch", op)
        ends = op in ("s_endpgm", "s_branch") or i + 1 == len(body)
        for j in ([] if ends else [i + 1]) + ([index[to]] if re.match(r"s_c?branch", op) else []):
            if j not in state or after & ~state[j]:
                state[j] = state.get(j, 0) | after
                todo.append(j)
    return [body[i][1] for i in sorted(state) if use[i] & state[i]]


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_accumulators_are_left_alone_until_the_wait(tmp_path):
    seen, grouped = 0, 0
    lib = capi.lib()._name
    for n, code in enumerate(_code_objects(open(lib, "rb").read())):
        if b"gemm_tiled_kernel" not in code:
            continue
        path = tmp_path / f"{n}.co"
        path.write_bytes(code)
        for name, body in _kernels(path):
            assert sum(t.startswith("v_mfma") for _, t, _ in body) > 0
            assert _touched_in_flight(body)[:4] == [], name
            seen += 1
            grouped += "Lb1ELb0ELb0ELi2E" in name or "Lb1ELb1ELb0ELi2E" in name
    assert seen > 100 and grouped == 11            # 8 of the FP8 experts, 3 of the GGUF experts
