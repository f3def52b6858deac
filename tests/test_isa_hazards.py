"""Wait states that the hardware leaves to software, checked in the disassembly of the library's own gfx950 kernels.

The compiler adds them for its own instructions and does not look into inline assembly, so a sequence written by hand has
to bring its own. The rules are those of the "manually inserted wait states" tables of AMD's CDNA instruction-set documents:
 - an SALU write of M0, then a load into LDS that takes its LDS address from M0: one wait state;
 - a VALU write of a vector register, then a data-parallel-primitive (DPP) read of it: two;
 - a VALU write of a vector register, then a matrix instruction that reads it: two.
"""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from lc0_amd import backend as be
from lc0_amd import build as lib_build

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
_REG = re.compile(r"(?<![\w.])([va])(?:(\d+)|\[(\d+):(\d+)\])")
_DPP = ("quad_perm", "row_shl", "row_shr", "row_ror", "row_mirror", "row_half_mirror", "row_bcast", "row_newbcast", "wave_")


def code_objects(library):
    """The gfx950 code objects bundled in a shared library."""
    data = open(library, "rb").read()
    out, at = [], data.find(_MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(_MAGIC))
        p = at + len(_MAGIC) + 8
        for _ in range(count if count < 64 else 0):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in triple and data[at + offset:at + offset + 4] == b"\x7fELF":
                out.append(data[at + offset:at + offset + size])
        at = data.find(_MAGIC, at + 1)
    return out


def disassemble(code_object):
    with tempfile.NamedTemporaryFile(suffix=".co") as f:
        f.write(code_object)
        f.flush()
        return subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", f.name], check=True,
                              capture_output=True, text=True).stdout


def _registers(operand):
    out = set()
    for kind, one, lo, hi in _REG.findall(operand):
        for r in range(int(one or lo), int(one or hi) + 1):
            out.add((kind, r))
    return out


def hazards(listing):
    """[(kernel, rule, first instruction, second instruction)] of a disassembly."""
    found, kernel, recent = [], "", []     # recent: (wait states since, instruction, M0 written, vector registers written)
    for line in listing.splitlines():
        if line.endswith(">:"):
            kernel, recent = line.split("<")[-1][:-2], []
            continue
        text = line.split("//")[0].strip()
        name, _, rest = text.partition(" ")
        if not re.match(r"[a-z]\w+$", name):
            continue
        ops = [o.strip() for o in rest.split(",")]
        is_mfma = name.startswith(("v_mfma", "v_smfmac"))
        reads = _registers(",".join(ops[1:])) if name.startswith("v_") else set()
        if name.startswith(("global_load_lds", "buffer_load")) and (name.startswith("global") or text.endswith(" lds")):
            found += [(kernel, "M0", i, text) for w, i, m0, _ in recent if m0 and w < 1]
        if is_mfma or any(d in rest for d in _DPP):
            rule = "matrix read" if is_mfma else "DPP read"
            # (DPP moves only the first source operand between lanes; the others are read like any operand)
            those = reads if is_mfma else _registers(re.sub(r"(quad_perm|row_\w+|bank_mask|wave_\w+).*", "", ops[1]))
            found += [(kernel, rule, i, text) for w, i, _, regs in recent if w < 2 and regs & those]
        states = int(ops[0], 0) + 1 if name == "s_nop" else 1
        recent = [(w + states, i, m0, regs) for w, i, m0, regs in recent if w + states < 2]
        written = set()
        if name.startswith("v_") and not is_mfma and not name.startswith(("v_cmp", "v_nop", "v_readlane", "v_readfirstlane")):
            written = _registers(ops[0])
            if "swap" in name:
                written |= _registers(ops[1])
        m0 = name.startswith("s_") and ops[0] == "m0"
        if written or m0:
            recent.append((0, text, m0, written))
    return found


LISTING = """
0000 <k>:
\ts_mov_b32 m0, s10
\t%s
\tglobal_load_lds_dwordx4 v[66:67], off
\tv_add_f32_e32 v5, v1, v2
\ts_nop 0
\t%s
\tv_mfma_f32_32x32x16_f16 v[16:31], v[2:5], v[6:9], v[16:31]
\tv_mov_b32_e32 v40, v1
\t%s
\tv_cndmask_b32_dpp v41, v40, v3, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf
"""


@pytest.mark.parametrize("fill,rules", [(("s_nop 0", "s_nop 0", "s_nop 1"), []), (("", "", "s_nop 0"),
                                                                                 ["M0", "matrix read", "DPP read"])])
def test_missing_wait_states_are_seen(fill, rules):
    assert [h[1] for h in hazards(LISTING % fill)] == rules


def test_no_kernel_of_the_library_lacks_a_wait_state():
    be.load_library()                       # (built on first use)
    objects = code_objects(lib_build.LIB)
    assert len(objects) >= 8                # one per source file with kernels
    missing, loads, products = [], 0, 0
    for o in objects:
        listing = disassemble(o)
        loads, products = loads + listing.count("global_load_lds"), products + listing.count("v_mfma")
        missing += hazards(listing)
    assert loads > 500 and products > 5000  # (the listing is what it is taken for)
    assert not missing, "%d, first: %s" % (len(missing), missing[:3])
