"""Wait states around the matrix instructions, and what their loops spill, in the machine code of the library as built.

The compiler keeps the distances that the hardware does not wait for by itself -- around its own MFMAs; those that are inline
assembly (recurrent_fwd_big.hpp, gemm16.hpp) it does not see inside.  What it puts between its own for gfx950, and what is
required of every v_mfma_f32_16x16x32_{f16,bf16} here, in wait states (an instruction is one, s_nop N is N + 1):

    8 from the MFMA to any other access to its result; none where an MFMA takes exactly that result as its own srcC;
    2 from a vector ALU instruction that writes a register (a copy between the halves of the register file, a spilled
      scalar) to the MFMA that reads it.

Every path of up to 8 wait states is followed, through branches too."""
import os
import re
import struct
import subprocess

import pytest

from fastlstm_amd import _lib

OBJDUMP, OBJCOPY = "/opt/rocm/llvm/bin/llvm-objdump", "/opt/rocm/llvm/bin/llvm-objcopy"
RESULT, OPERAND = 8, 2
MFMA = ("v_mfma_f32_16x16x32_f16", "v_mfma_f32_16x16x32_bf16")
REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))")


def code_objects(path, tmp):
    fat = os.path.join(tmp, "fatbin")
    subprocess.run([OBJCOPY, "--dump-section", ".hip_fatbin=" + fat, path, os.devnull], check=True)
    data, magic, at = open(fat, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        (count,), p = struct.unpack_from("<Q", data, at + len(magic)), at + len(magic) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n] and size:
                yield data[at + off:at + off + size]
            p += 24 + n
        at += len(magic)


def registers(text):
    """One bit per register named: v in the lower 512, a in the upper."""
    bits = 0
    for half, lo, hi, one in REG.findall(text):
        lo, hi = (int(lo), int(hi)) if lo else (int(one), int(one))
        bits |= ((1 << (hi - lo + 1)) - 1) << (lo + (512 if half == "a" else 0))
    return bits


def parse(lines):
    """{function: [(text, opcode, wait states, all registers, (dst, srcA|srcB, srcC) of an MFMA, written by the vector ALU,
    branch target or None, falls through)]}"""
    functions, current, address = {}, None, {}
    for line in lines:
        head = re.match(r"^[0-9a-f]+ <(.+)>:$", line)
        if head:
            current = functions.setdefault(head.group(1), [])
            continue
        m = re.match(r"^\s+(\S+)(?: (.*?))?\s*// ([0-9A-F]+):.*?(?:<.+\+0x([0-9a-f]+)>|<[^+>]+>)?$", line)
        if not m or current is None:
            continue
        op, args, pc = m.group(1), m.group(2) or "", int(m.group(3), 16)
        if not current:
            address[id(current)] = pc
        wait = int(args, 0) + 1 if op == "s_nop" else 1
        parts = re.split(r",\s*(?![^\[]*\])", args) if args else []
        mfma = alu = None
        if op in MFMA:
            regs = [registers(a) for a in parts[:4]]
            mfma = (regs[0], regs[1] | regs[2], regs[3])
        elif op.startswith("v_") and parts:
            alu = registers(parts[0])
        target = pc_target = None
        if op.startswith(("s_branch", "s_cbranch")):
            pc_target = address[id(current)] + int(m.group(4) or "0", 16)
        current.append([pc, op + " " + args, op, wait, registers(args), mfma, alu, pc_target,
                        not op.startswith(("s_branch", "s_endpgm", "s_setpc"))])
    return functions


def violations(code):
    index = {ins[0]: k for k, ins in enumerate(code)}
    bad = []

    def follow(start, regs, limit, clash):
        seen, todo = {}, [(start, 0)]
        while todo:
            k, passed = todo.pop()
            while k < len(code) and passed < limit and seen.get(k, limit) > passed:
                seen[k] = passed
                ins = code[k]
                if clash(ins, regs):
                    bad.append((code[start - 1][1], ins[1], passed))
                    return
                passed += ins[3]
                if ins[7] is not None:
                    todo.append((index[ins[7]], passed))
                if not ins[8]:
                    break
                k += 1

    def touches_result(ins, regs):
        if ins[5]:
            dst, ab, c = ins[5]
            return bool(ab & regs) or (bool(c & regs) and c != regs)   # (MFMAs write in order)
        return bool(ins[4] & regs)

    def reads_operand(ins, regs):
        return bool(ins[5]) and bool((ins[5][1] | ins[5][2]) & regs)

    for k, ins in enumerate(code):
        if ins[5]:
            follow(k + 1, ins[5][0], RESULT, touches_result)
        elif ins[6]:
            follow(k + 1, ins[6], OPERAND, reads_operand)
    return bad


def scratch_in_matrix_loops(code):
    """Scratch accesses in the innermost loops that hold MFMAs: [(first pc, MFMAs, accesses)]."""
    index = {ins[0]: k for k, ins in enumerate(code)}
    loops = [(index[ins[7]], k) for k, ins in enumerate(code) if ins[7] is not None and ins[7] <= ins[0]]
    found = []
    for a, b in loops:
        if any((c, d) != (a, b) and a <= c and d <= b for c, d in loops):
            continue
        mfma, scratch = (sum(ins[2].startswith(what) for ins in code[a:b + 1]) for what in ("v_mfma", "scratch_"))
        if mfma and scratch:
            found.append((code[a][0], mfma, scratch))
    return found


def kernels_of(path, tmp):
    for n, blob in enumerate(code_objects(path, str(tmp))):
        if b"lstm_" not in blob and b"gemm" not in blob:
            continue
        name = os.path.join(str(tmp), "co%d" % n)
        open(name, "wb").write(blob)
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", name], check=True, capture_output=True, text=True).stdout
        for fn, code in parse(text.splitlines()).items():
            yield fn, code


def test_the_check_sees_what_it_looks_for():
    def listing(*body):
        return parse(["0000000000000000 <k>:"] + ["\t%s // %012X: 00000000" % (b, 8 * i) for i, b in enumerate(body)])["k"]

    mfma = "v_mfma_f32_16x16x32_f16 v[0:3], a[0:3], v[8:11], v[0:3]"
    read = "ds_write_b128 v20, v[0:3]"
    assert not violations(listing(mfma, mfma, "s_nop 7", read))
    assert violations(listing(mfma, "s_nop 6", read))                       # one short
    assert violations(listing(mfma, "v_mov_b32_e32 v30, v2", "s_nop 7", read))   # a copy in between
    assert violations(listing(mfma, "s_nop 6", "v_mfma_f32_16x16x32_f16 v[4:7], v[0:3], v[8:11], v[4:7]"))
    assert violations(listing("v_accvgpr_write_b32 a2, v9", "s_nop 0", mfma))
    assert not violations(listing("v_accvgpr_write_b32 a2, v9", "s_nop 1", mfma))
    back = parse(["0000000000000000 <k>:", "\t%s // 000000000000: 00000000" % read, "\t%s // 000000000008: 00000000" % mfma,
                  "\ts_branch 65533 // 000000000010: 00000000 <k+0x0>"])["k"]
    assert violations(back)                                                 # round a loop


def test_the_scratch_check_sees_what_it_looks_for():
    def listing(*body):
        return parse(["0000000000000000 <k>:"] + ["\t%s // %012X: 00000000%s" % (b, 8 * i, t) for i, (b, t) in enumerate(body)])["k"]

    mfma = ("v_mfma_f32_16x16x32_f16 v[0:3], a[0:3], v[8:11], v[0:3]", "")
    load, back = ("scratch_load_dwordx4 v[0:3], off, off", ""), ("s_cbranch_scc1 65530", " <k+0x8>")
    assert scratch_in_matrix_loops(listing(load, mfma, load, back)) == [(8, 1, 1)]
    assert not scratch_in_matrix_loops(listing(load, mfma, back, load))


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    """(kernel, wait states broken, scratch accesses in its matrix loops) of every kernel with MFMAs."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    return [(fn, violations(code), scratch_in_matrix_loops(code))
            for fn, code in kernels_of(_lib.LIB_PATH, tmp_path_factory.mktemp("code")) if any(ins[2].startswith("v_mfma") for ins in code)]


def test_distances_around_the_matrix_instructions(built):
    assert sum("_big_kernel" in fn for fn, _, _ in built) == 80 and len(built) > 100
    for fn, broken, _ in built:
        assert not broken, (fn, broken[:3])


def test_matrix_loops_stay_out_of_scratch(built):
    """Accumulators moved to scratch and back in every pass of a k loop: the reverse launch with weight gradients took four
    times as long at 256 <= H <= 512.  (The step loops hold no loop inside and are innermost ones too.)"""
    spilling = [(fn, s) for fn, _, s in built if s]
    assert not spilling, spilling
