"""The Dense kernels' matrix instructions are written as assembly (csrc/dt_dense_kernel.h), which the compiler knows nothing of: it
does not keep other instructions off their results until these are there.  What it made of the library's kernels is read back and
checked: between a matrix instruction and the pair of s_nop behind the K loop, along every path, nothing but matrix
instructions touches a sum, and no vector instruction writes an operand right in front of the one that reads it."""
import os
import re
import shutil
import struct
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "..", "draw-things-community_amd", "libdthip.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MFMA = "v_mfma_f32_16x16x32_f16"
RANGE = re.compile(r"\bv(?:(\d+)|\[(\d+):(\d+)\])")


def registers(text):
    """The vector registers named in `text`."""
    out = set()
    for one, lo, hi in RANGE.findall(text):
        out.update(range(int(lo), int(hi) + 1) if lo else (int(one),))
    return out


def zero(code, i):
    """Whether the move at i sets registers to zero, itself or from registers that a move before it set."""
    source = code[i][1].split(", ", 1)[1]
    if not registers(source):
        return source == "0"
    for j in range(i - 1, max(i - 100, -1), -1):
        text = code[j][1]
        if text.startswith("v_") and registers(text.split(",")[0]) & registers(source):
            return text.startswith("v_mov_b") and zero(code, j)
    return False


def faults(code):
    """code: [(address, text, address of a branch's target or None)].  The instructions that get in the way of a sum or an operand,
    and the number of matrix instructions."""
    at = {addr: i for i, (addr, _, _) in enumerate(code)}
    mfma = [i for i, (_, text, _) in enumerate(code) if text.startswith(MFMA)]
    sums = set().union(*(registers(code[i][1].split(",")[0]) for i in mfma))
    settled = {i for i in range(len(code) - 1) if code[i][1] == code[i + 1][1] == "s_nop 15"}
    # Sums set to zero: a loop begins.  (The waves that stage weights have a loop of their own; none runs both, which the
    # branches between them do not show.)
    begins = {i for i, (_, text, _) in enumerate(code)
              if text.startswith("v_mov_b") and registers(text.split(",")[0]) <= sums and zero(code, i)}

    def follow(i):
        _, text, target = code[i]
        if target is not None:
            yield at[target]
        if not text.startswith(("s_endpgm", "s_branch")) and i + 1 < len(code):
            yield i + 1

    def reach(todo, step, stop):
        seen = set()
        while todo:
            i = todo.pop()
            if i not in seen and i not in stop:
                seen.add(i)
                todo.extend(step(i))
        return seen

    before = {}
    for i in range(len(code)):
        for j in follow(i):
            before.setdefault(j, []).append(i)
    in_flight = reach(list(mfma), follow, settled | begins)
    # ... of these, what leads on to a matrix instruction or to the end without a loop's beginning
    ends = [j for i in settled for j in before.get(i, [])] + [i for i, (_, text, _) in enumerate(code) if text == "s_endpgm"]
    in_flight &= reach(mfma + ends, lambda i: before.get(i, []), begins | settled)
    bad = []
    for i in sorted(in_flight):
        text = code[i][1]
        if text.startswith(MFMA):
            for _, earlier, _ in code[max(0, i - 2):i]:
                if earlier.startswith("v_") and not earlier.startswith("v_mfma") and registers(earlier.split(",")[0]) & registers(text):
                    bad.append((earlier, text))
        elif text.startswith(("v_", "ds_", "global_", "buffer_", "flat_", "scratch_")) and registers(text) & sums:
            bad.append((text,))
    return bad, len(mfma)


def device_code(path):
    """The gfx950 code objects that the library carries."""
    blob, magic, i = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (i := blob.find(magic, i)) >= 0:
        count, at = struct.unpack_from("<Q", blob, i + len(magic))[0], i + len(magic) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, at)
            if b"gfx950" in blob[at + 24:at + 24 + n]:
                yield blob[i + off:i + off + size]
            at += 24 + n
        i += len(magic)


def kernels(obj, name, tmp_path):
    """(symbol, code) of the kernels of a code object whose symbols contain `name`."""
    if name.encode() not in obj:
        return
    path = tmp_path / "code.o"
    path.write_bytes(obj)
    listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
    symbol, base, code = None, 0, []
    for line in listing.split("\n"):
        if line and line[0] in "0123456789abcdef" and line.endswith(">:"):
            if symbol and name in symbol:
                yield symbol, code
            base, symbol, code = int(line.split()[0], 16), line.split("<")[1][:-2], []
        elif line.startswith("\t") and symbol and name in symbol:
            text, _, note = line.strip().partition("//")
            if not note:  # (padding)
                continue
            target = re.search(r"\+0x([0-9a-f]+)>", note) if "branch" in text else None
            begins = text.startswith(("s_branch", "s_cbranch")) and f"<{symbol}>" in note
            code.append((int(note.split(":")[0], 16), text.strip(), base + int(target.group(1), 16) if target else base if begins else None))
    if symbol and name in symbol:
        yield symbol, code


def test_the_check_sees_what_it_is_for():
    loop = [f"{MFMA} v[4:7], v[20:23], v[24:27], v[4:7]", "ds_read_b128 v[20:23], v1", f"{MFMA} v[8:11], v[20:23], v[24:27], v[8:11]",
            "s_cbranch_scc1", "s_nop 15", "s_nop 15", "v_mov_b32_e32 v4, v8", "s_endpgm"]
    made = lambda lines: [(4 * i, t, 0 if t == "s_cbranch_scc1" else None) for i, t in enumerate(lines)]
    assert faults(made(loop)) == ([], 2)
    for place, planted in ((1, "v_mov_b32_e32 v30, v5"), (4, "v_accvgpr_write_b32 a0, v9"), (3, "scratch_store_dwordx4 off, v[8:11], off"),
                           (2, "v_add_u32_e32 v22, v1, v2")):
        text = loop[:place] + [planted] + loop[place:]
        assert faults(made(text))[0], planted
    assert faults(made(loop[:4] + loop[5:]))[0]  # one s_nop short


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_nothing_touches_the_sums_of_the_dense_kernels(tmp_path):
    assert os.path.exists(LIB), "build first"
    checked = 0
    for obj in device_code(LIB):
        for symbol, code in kernels(obj, "dense_qx_kernel", tmp_path):
            bad, n = faults(code)
            assert n > 0 and not bad, (symbol, bad[:4])
            checked += 1
    assert checked >= 100
