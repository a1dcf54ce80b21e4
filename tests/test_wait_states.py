"""Wait states that the hardware does not keep by itself, in the built library's own code: the compiler pads its instructions with
them, but puts none inside an inline assembly statement, and counts no instruction in one as a use.  From one instruction to the next that
uses its result, counted in instructions issued between (s_nop n counts n + 1):

- mask: a vector instruction that writes a mask or another scalar register, to a vector instruction that reads it: 2
- address: the same, to a memory instruction: 5
- transcendental: such an instruction, to a vector instruction of another kind that reads its result: 1
- matrix: a matrix instruction, to a vector instruction or a store that reads its result: its passes and 4.  The compiler takes some
  branches out again that it has counted, so 2 fewer are let pass here.
"""
import os
import re
import struct
import subprocess
from concurrent.futures import ProcessPoolExecutor

import pytest

from conftest import PKG

LIB = os.path.join(PKG, "lib", "libmpsa.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
REG = re.compile(r"\b([vsa])(?:\[(\d+):(\d+)\]|(\d+))|\bvcc")
TRANS = ("v_exp_", "v_log_", "v_rcp_", "v_rsq_", "v_sqrt_", "v_sin_", "v_cos_")
MEMORY = ("global_", "buffer_", "flat_", "scratch_")
TWO_RESULTS = ("v_add_co", "v_addc", "v_sub_co", "v_subb", "v_subrev_co", "v_mad_u64", "v_mad_i64", "v_div_scale")


def registers(operand):
    out = []
    for m in REG.finditer(operand):
        kind, first, last, one = m.groups()
        if kind is None:
            out.append("vcc")
        else:
            out += [(kind, i) for i in (range(int(first), int(last) + 1) if first else (int(one),))]
    return out


def passes(op, rest):
    both4 = "cbsz:4" in rest and "blgp:4" in rest
    if "f8f6f4" in op:
        return (8 if "32x32" in op else 4) * (1 if both4 else 2)
    return {"32x32x16": 8, "16x16x32": 4}[op.split("_")[3]]


def too_close(text):
    """(rule, kernel, instruction, instruction that comes too early, wait states between) of a code object's disassembly; read from
    top to bottom, so along the paths that take no branch."""
    bad, kernel, now, last = [], None, 0, {}
    for line in text.splitlines():
        if line.endswith(">:"):
            kernel, last = line.split("<")[1][:-2], {}
            continue
        line = line.split("//")[0].strip()
        op, _, rest = line.partition(" ")
        if kernel is None or not op or ":" in op:
            continue
        if op == "s_nop":
            now += int(rest, 0) + 1
            continue
        if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
            last = {}
            continue
        operands = re.split(r",\s*(?![^\[]*\])", rest)
        vector, matrix = op.startswith("v_"), op.startswith("v_mfma")
        if vector or op.startswith(MEMORY):
            results = 0 if not vector else 2 if op.startswith(TWO_RESULTS) or "swap" in op else 1
            read = {r for o in operands[0 if "swap" in op else results:] for r in registers(o)}
            for r in read & last.keys():
                at, rule, states, by = last[r]
                if rule == "mask" and not vector:
                    rule = "address"
                wanted = {"mask": 2, "address": 5, "transcendental": 1 if vector and not op.startswith(TRANS) else 0,
                          "matrix": 0 if matrix or not (vector or "store" in op) else states}[rule]
                if now - at - 1 < wanted:
                    bad.append((rule, kernel, by, line, now - at - 1))
            for r in (r for o in operands[:results] for r in registers(o)):
                last.pop(r, None)
                if r == "vcc" or r[0] == "s":
                    last[r] = (now, "mask", 0, line)
                elif matrix:
                    last[r] = (now, "matrix", passes(op, rest) + 2, line)
                elif op.startswith(TRANS):
                    last[r] = (now, "transcendental", 0, line)
        elif op.startswith("s_") and not op.startswith(("s_cmp", "s_bitcmp", "s_cbranch", "s_waitcnt")):
            for r in registers(operands[0]):
                last.pop(r, None)
        now += 1
    return bad


def check(code, path):
    with open(path, "wb") as f:
        f.write(code)
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", path], check=True, capture_output=True, text=True).stdout
    return text.count(">:"), too_close(text)


def code_objects(data):
    """The gfx950 objects of a library's offload bundles."""
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length] and size:
                yield data[at + offset:at + offset + size]
            p += 24 + length
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and the ROCm disassembler")
    with open(LIB, "rb") as f:
        objects = sorted(code_objects(f.read()), key=len, reverse=True)
    d = tmp_path_factory.mktemp("objects")
    with ProcessPoolExecutor(4) as pool:
        done = list(pool.map(check, objects, [str(d / f"{i}.co") for i in range(len(objects))]))
    assert sum(n for n, _ in done) > 100          # kernels
    return [b for _, found in done for b in found]


@pytest.mark.parametrize("rule", ["mask", "address", "transcendental", "matrix"])
def test_no_result_is_used_too_early(library, rule):
    bad = [b[1:] for b in library if b[0] == rule]
    assert not bad, (len(bad), bad[:4])


@pytest.mark.parametrize("between, states", [("", 0), ("\ts_mov_b32 s3, 8\n", 1), ("\ts_nop 1\n", 2)])
def test_masks_in_a_listing(between, states):
    found = too_close("0000000000001900 <kernel>:\n\tv_cmp_ge_i32_e32 vcc, s3, v66\n" + between + "\tv_cndmask_b32_e32 v51, v51, v67, vcc\n")
    assert [b[4] for b in found] == ([states] if states < 2 else [])


@pytest.mark.parametrize("states", [0, 4, 5])
def test_addresses_in_a_listing(states):
    found = too_close("0000000000001900 <kernel>:\n\tv_readfirstlane_b32 s7, v5\n" + "\ts_nop 0\n" * states + "\tglobal_load_lds_dwordx4 v8, s[6:7]\n")
    assert [(b[0], b[4]) for b in found] == ([("address", states)] if states < 5 else [])


@pytest.mark.parametrize("op, formats, states", [("v_mfma_f32_32x32x16_bf16", "", 12), ("v_mfma_scale_f32_32x32x64_f8f6f4", " cbsz:4 blgp:4", 12),
                                                 ("v_mfma_scale_f32_32x32x64_f8f6f4", " cbsz:4", 20), ("v_mfma_scale_f32_32x32x64_f8f6f4", "", 20)])
def test_products_in_a_listing(op, formats, states):
    listing = "0000000000001900 <kernel>:\n\t" + op + " v[0:15], v[32:39], v[40:47], v[0:15]" + formats + "\n\ts_nop 7\n\ts_nop %d\n\tv_exp_f32_e32 v16, v15\n"
    assert not too_close(listing % (states - 9)) and not too_close(listing % (states - 11)) and [b[4] for b in too_close(listing % (states - 12))] == [states - 3]
