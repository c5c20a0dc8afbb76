"""The device code of the built library against a hardware rule that the compiler does not
apply to inline assembly: a vector-memory instruction reads a scalar register that a VALU
instruction (a spilled register's v_readlane, a v_readfirstlane) wrote only five wait states
or more after that write.  The LDS DMA statements of gemm_common.h and attention.hip take
their base in scalar registers; a base read too early would send the load elsewhere."""
import re
import shutil
import struct
import subprocess

import pytest

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
WAIT_STATES = 5
_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
_SGPR = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b")


def _code_objects(blob: bytes):
    """The gfx950 code objects of a library's offload bundles."""
    at = blob.find(_MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            target = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if size and target.endswith(b"gfx950"):
                yield blob[at + off:at + off + size]
        at = blob.find(_MAGIC, at + 24)


def _sgprs(text: str):
    out = set()
    for lo, hi, one in _SGPR.findall(text):
        out.update([int(one)] if one else range(int(lo), int(hi) + 1))
    return out


def hazards(lines):
    """(kernel, write, read, wait states between) of every vector-memory instruction that
    reads a scalar register too soon after a VALU write, in listing order."""
    kernel, recent, found = "", [], []   # recent: (wait states, registers written, text)
    for line in lines:
        s = line.split("//")[0].strip()
        if not s:
            continue
        if s.endswith(":"):
            kernel, recent = s, []
            continue
        op, _, args = s.partition(" ")
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            waited, reads = 0, _sgprs(args)
            for states, wrote, text in reversed(recent):
                if waited >= WAIT_STATES:
                    break
                if wrote & reads:
                    found.append((kernel, text, s, waited))
                    break
                waited += states
        states = int(args.strip(), 0) + 1 if op == "s_nop" else 1
        wrote = set()
        if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")):
            wrote = _sgprs(args.split(",")[0])
        elif re.match(r"v_(add|sub|addc|subb|subrev|subbrev)_co_|v_div_scale|v_mad_[ui]64", op):
            wrote = _sgprs(args.split(",")[1])
        recent = (recent + [(states, wrote, s)])[-WAIT_STATES - 1:]
    return found


@pytest.mark.parametrize("between,safe", [
    ([], False),
    (["s_mov_b32 m0, s4", "s_nop 0"], False),
    (["s_mov_b32 m0, s4", "s_nop 2"], False),
    (["s_mov_b32 m0, s4", "s_nop 3"], True),
    (["v_add_u32_e32 v1, v2, v3"] * 5, True),
])
def test_the_check_counts_wait_states(between, safe):
    code = ["0000 <k>:", "v_readlane_b32 s7, v9, 3", *between,
            "global_load_lds_dword v2, s[6:7]"]
    assert (hazards(code) == []) == safe
    # another register's write is no hazard
    code[1] = "v_readlane_b32 s8, v9, 3"
    assert hazards(code) == []


def test_scalar_bases_of_vector_memory_settle(g5lib, tmp_path):
    from genet5_amd import _lib
    objs = list(_code_objects(_lib.LIB_PATH.read_bytes()))
    assert objs, "no gfx950 code object in the library"
    loads = 0
    for i, obj in enumerate(objs):
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        lines = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True,
                               check=True).stdout.splitlines()
        loads += sum("global_load_lds" in line for line in lines)
        assert hazards(lines) == []
    assert loads > 0, "no LDS DMA found in the disassembly"
