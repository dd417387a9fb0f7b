"""The lane masks of the compiled kernels, read from the built library's own
code objects.

When a loop ends that each lane leaves by itself, no lane is active until the
mask of an enclosing region is restored.  The compiler may drop the mask
restore right after the loop, where another one follows, and later place
reloads of spilled vector registers in between: they then load nothing and the
register keeps what the loop left in it.  A right-hand-side kernel with the
mirror pass of bssn_edge_lds.h written as such a loop had wrong A_xz values by
it.  No kernel may hold a vector write there, and the mirror pass, whose trip
count is the same for every lane, must not be such a loop.
"""
import os
import re
import shutil
import struct
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "..", "nr-amssncku_amd", "amssbssn", "libamssbssn.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
LINE = re.compile(r"^\t(\S+)(?: (.*?))?\s*// ([0-9A-F]+):(?:.*<(\S+?)(?:\+0x([0-9a-f]+))?>)?")
LOOP_END = re.compile(r"exec, exec, ")
VECTOR = re.compile(r"v_(?!cmp|readlane|readfirstlane|writelane)|ds_read|(scratch|global|buffer|flat)_load_d")


def _code_objects(path):
    d = open(path, "rb").read()
    i = d.find(MAGIC)
    while i >= 0:
        (count,) = struct.unpack_from("<Q", d, i + len(MAGIC))
        p = i + len(MAGIC) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", d, p)
            if b"gfx950" in d[p + 24:p + 24 + n]:
                yield d[i + off:i + off + size]
            p += 24 + n
        i = d.find(MAGIC, i + len(MAGIC))


def _kernels(text):
    """name -> [(address, mnemonic, operands, branch target)] of a disassembly"""
    base, kernels, cur = {}, {}, None
    for line in text.splitlines():
        if line.endswith(">:"):
            addr, name = line.split()
            base[name[1:-2]] = int(addr, 16)
            cur = kernels.setdefault(name[1:-2], [])
            continue
        m = LINE.match(line)
        if m and cur is not None:
            to = (m[4], int(m[5] or "0", 16)) if m[4] else None
            cur.append((int(m[3], 16), m[1], m[2] or "", to))
    return {k: [(a, op, r, base[t[0]] + t[1] if t else None) for a, op, r, t in ins] for k, ins in kernels.items()}


def lane_loops(ins):
    """indexes of the branches that follow a loop's s_andn2_b64 exec, exec"""
    return [i + 1 for i, (_, op, r, _) in enumerate(ins[:-1])
            if op == "s_andn2_b64" and LOOP_END.match(r) and ins[i + 1][1] in ("s_cbranch_execz", "s_cbranch_execnz")]


def lost_writes(ins):
    """vector writes between the end of a loop and the next write of exec"""
    at = {x[0]: i for i, x in enumerate(ins)}
    lost = []
    for b in lane_loops(ins):
        i = at[ins[b][3]] if ins[b][1] == "s_cbranch_execz" else b + 1
        while i < len(ins):
            _, op, r, to = ins[i]
            if r.startswith("exec") or "saveexec" in op or op == "s_endpgm" or op.startswith("s_cbranch"):
                break
            if op == "s_branch":
                i = at[to]
                continue
            if VECTOR.match(op):
                lost.append("%x: %s %s" % (ins[i][0], op, r))
            i += 1
    return lost


def test_the_check_finds_a_reload_after_a_loop():
    asm = ("0000000000000000 <k>:\n"
           "\ts_andn2_b64 exec, exec, s[40:41]      // 000000000000: 00\n"
           "\ts_cbranch_execz 2                     // 000000000004: 00 <k+0xc>\n"
           "\ts_branch 65535                        // 000000000008: 00 <k+0x0>\n"
           "\ts_barrier                             // 00000000000C: 00\n"
           "\tscratch_load_dwordx2 v[208:209], off, off offset:544 // 000000000010: 00\n"
           "\ts_or_b64 exec, exec, s[42:43]         // 000000000018: 00\n"
           "\tv_mul_f64 v[20:21], v[208:209], v[162:163] // 00000000001C: 00\n")
    ins = _kernels(asm)["k"]
    assert lost_writes(ins) == ["10: scratch_load_dwordx2 v[208:209], off, off offset:544"]
    assert lost_writes(ins[:4] + ins[5:]) == []


@pytest.mark.skipif(not os.path.exists(LIB) or shutil.which(OBJDUMP) is None, reason="needs the built library")
def test_no_kernel_writes_a_vector_register_while_no_lane_is_active(tmp_path):
    kernels, mirror = 0, 0
    for n, co in enumerate(_code_objects(LIB)):
        f = tmp_path / ("%d.co" % n)
        f.write_bytes(co)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True,
                              text=True).stdout
        for name, ins in _kernels(text).items():
            kernels += len(ins) > 0
            assert not lost_writes(ins), (name, lost_writes(ins))
            if re.search(r"rhs_edge_lds_kernelILi\dELb\dELb\dELb1EE", name):  # <GAUGE, CO, ODD, MIRROR = true>
                mirror += 1
                assert not lane_loops(ins), name
    assert kernels > 100 and mirror == 8
